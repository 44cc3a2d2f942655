"""Resident launches that the gate refuses (with gate polls set to 0 it never opens, as if other work
kept a block off the device): their steps are taken by stage launches, with the same bits, whatever
was asked of the model before anyone waited.  With ring polls at 0 as well a launch that did go in
would end in an error."""
import ctypes

import numpy as np
import pytest

import self_amd
from self_amd import call
from tests.test_gpu_resident_giveup import gives_up, model

pytestmark = pytest.mark.gpu


def refuse(m, on=True):
    m._param(self_amd.PARAM_POLLS, 0 if on else 1 << 26)
    m._param(self_amd.PARAM_GATE_POLLS, 0 if on else 4096)


def enqueue(m, steps, dt):
    call("selfamd_model2d_forward_step", m._h, steps, float(dt))


def stages(m, steps, dt):
    for _ in range(steps):
        for st in range(3):
            m.Stage(st, dt)


CASES = [("sw", 7, 10, 10, "affine", 0), ("sw", 5, 11, 13, "nodal", 0), ("lsw", 6, 45, 37, "affine", 0),
         ("euler", 4, 73, 61, "affine", 0), ("sw", 3, 33, 31, "affine", 128)]


@pytest.mark.parametrize("kind,N,nx,ny,metrics,hidden", CASES)
def test_refused_steps_are_taken(kind, N, nx, ny, metrics, hidden):
    c, m = model(kind, N, nx, ny, metrics, hidden)
    dt = c.dt(0.05)
    calls = [(5, dt), (2, dt), (2, dt), (1, dt), (3, 0.5 * dt), (2, dt)]
    for n, d in calls:
        stages(m, n, d)
    want, want_t = m.solution, m.t
    stages(m, 2, dt)
    after = m.solution
    # one call after another, waiting for each
    m.SetSolution(c.sol)
    refuse(m)
    for n, d in calls:
        m.ForwardStep(n, d)
    np.testing.assert_array_equal(m.solution, want)
    # without waiting: the launches after a refused one end at once as well (a new model, which
    # does not keep to step graphs yet)
    c, m = model(kind, N, nx, ny, metrics, hidden)
    refuse(m)
    for n, d in calls:
        enqueue(m, n, d)
    np.testing.assert_array_equal(m.solution, want)
    assert m.t == want_t
    stages(m, 2, dt)  # traces and lagged velocities
    np.testing.assert_array_equal(m.solution, after)


def test_readers_and_changes_see_the_steps_taken():
    """Everything that reads the state or changes what the steps depend on, right after a call that is
    refused."""
    _, r = model("sw", 3, 9, 8)
    c, _ = model("sw", 3, 9, 8)
    dt = c.dt(0.05)
    field = 0.01 * np.ones((72, 4, 4))
    value = self_amd.DeviceArray((1,), zero=True)

    def noalloc(m):
        call("selfamd_model2d_integral_noalloc", m._h, 2, value.ptr)
        self_amd.synchronize()
        return value.to_host()[0]

    actions = [lambda m: m.solution, lambda m: m.CalculateTendency(), lambda m: m.flux_registers()[0], noalloc,
               lambda m: m.CalculateEntropy(), lambda m: (m.Stage(0, dt), m.Stage(1, dt), m.Stage(2, dt), m.solution)[3],
               lambda m: (m.SetTopography(field), m.ForwardStep(1, dt), m.solution)[2],
               lambda m: (m._param(self_amd.PARAM_G, 2.0), m.ForwardStep(1, dt), m.solution)[2],
               lambda m: (m.SetNodalMetrics(True), m.ForwardStep(1, dt), m.solution)[2],
               lambda m: (m.SetBands(2), m.ForwardStep(1, dt), m.solution)[2],
               lambda m: (m.time_steps(4, dt), m.solution)[1],
               lambda m: (m.SetSolution(c.sol), m.ForwardStep(3, dt), m.solution)[2]]

    def scattered(m):
        b = self_amd.Batch([m], [dt])
        b.ForwardStep(2)
        b.scatter()
        return m.solution
    actions.append(scattered)
    for k, action in enumerate(actions):
        out = []
        for on in (False, True):
            _, m = model("sw", 3, 9, 8)
            if on:
                refuse(m)
                enqueue(m, 4, dt)
            else:
                stages(m, 4, dt)
            out.append(action(m))
        np.testing.assert_array_equal(out[0], out[1], err_msg=str(k))


def test_scatter_over_refused_steps():
    c, m = model("sw", 5, 9, 9)
    dt = c.dt(0.05)
    batch = self_amd.Batch([m], [dt])
    batch.ForwardStep(3)
    batch.scatter()
    want = m.solution
    refuse(m)
    enqueue(m, 4, dt)
    batch.scatter()
    np.testing.assert_array_equal(m.solution, want)
    stages(m, 4, dt)
    want = m.solution
    batch.scatter()
    refuse(m, False)
    m.ForwardStep(4, dt)
    np.testing.assert_array_equal(m.solution, want)


def test_the_network_may_change_in_stream_order():
    c, m = model("sw", 3, 33, 31, hidden=128)
    dt = c.dt(0.05)
    net = m.net
    stages(m, 4, dt)
    want = m.solution
    m.SetSolution(c.sol)
    refuse(m)
    stream = ctypes.c_void_p()
    call("selfamd_model2d_stream", m._h, ctypes.byref(stream))
    X = self_amd.DeviceArray.from_host(np.ones((64, net.nIn), np.float32))
    T = self_amd.DeviceArray.from_host(np.ones((64, net.nOut), np.float32))
    enqueue(m, 4, dt)
    call("selfamd_mlp_loss_grad", net._h, X.ptr, T.ptr, 64, None, stream)
    call("selfamd_mlp_adam_step", net._h, 0.1, 1, stream)
    np.testing.assert_array_equal(m.solution, want)


def test_a_refused_model_comes_back():
    """After a refused launch 64 calls take step graphs; then launches go in again."""
    c, m = model("sw", 3, 9, 8)
    dt = c.dt(0.05)
    refuse(m)
    m.ForwardStep(2, dt)
    m._param(self_amd.PARAM_GATE_POLLS, 4096)
    for _ in range(64):
        m.ForwardStep(2, dt)
    assert gives_up(m, 2, dt)
    refuse(m, False)
    m.SetSolution(c.sol)
    m.ForwardStep(5, dt)
    got = m.solution
    m.SetSolution(c.sol)
    stages(m, 5, dt)
    np.testing.assert_array_equal(got, m.solution)
