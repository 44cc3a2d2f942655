"""Resident launches whose waits give up (a limit of no polls at all, set from the host: every
block runs to its end without its neighbours): the error that every reader of the state reports,
and the ways back to a valid state.  The same limit shows which calls run as resident launches."""
import ctypes

import numpy as np
import pytest

import self_amd
from self_amd import SelfAmdError, call
from tests.cases import Case

pytestmark = pytest.mark.gpu

POLLS = self_amd.PARAM_POLLS


def model(kind, N, nx, ny, metrics="affine", hidden=0):
    c = Case(kind, N, nx, ny, bcid=self_amd.BC_NONORMALFLOW, metrics=metrics)
    m, _ = c.gpu_model()
    if hidden:
        rng = np.random.default_rng(hidden)
        n_out = m.shape[1] * (N + 1) ** 2
        n_in = n_out + 3
        m.net = self_amd.MLP(n_in, hidden, n_out, nx * ny)
        m.net.set_params({k: 0.1 * rng.standard_normal(s) for k, s in m.net._shapes().items()})
        m.SetClosure(m.net, np.zeros(n_in, np.float32), np.ones(n_in, np.float32), np.zeros(n_out, np.float32),
                     np.full(n_out, 1e-3, np.float32))
    return c, m


def gives_up(m, steps, dt):
    """Whether a call of `steps` steps runs as a resident launch."""
    m._param(POLLS, 0)
    try:
        m.ForwardStep(steps, dt)  # waits for the steps
        return False
    except SelfAmdError as e:
        assert "gave up" in str(e)
        return True


@pytest.mark.parametrize("kind,N,nx,ny,metrics,hidden,steps,resident", [
    ("lsw", 7, 10, 10, "affine", 0, 2, True), ("lsw", 7, 10, 10, "affine", 0, 1, False),
    ("sw", 3, 64, 64, "affine", 0, 1, True), ("sw", 7, 64, 64, "affine", 0, 5, True),
    ("sw", 7, 81, 64, "affine", 0, 5, False),  # more blocks than the device holds
    ("sw", 5, 11, 13, "nodal", 0, 5, True), ("sw", 2, 4, 3, "nodal", 0, 5, True), ("lsw", 1, 30, 30, "affine", 0, 5, True),
    ("euler", 4, 73, 61, "affine", 0, 5, True), ("euler", 7, 6, 5, "nodal", 0, 5, True),
    ("sw", 3, 64, 64, "affine", 128, 1, True), ("euler", 4, 8, 6, "affine", 64, 2, True),
    ("sw", 3, 8, 8, "affine", 129, 5, False), ("sw", 5, 8, 8, "affine", 64, 5, False),
    ("sw", 3, 8, 8, "nodal", 0, 5, True),
])
def test_which_calls_are_resident(kind, N, nx, ny, metrics, hidden, steps, resident):
    c, m = model(kind, N, nx, ny, metrics, hidden)
    assert gives_up(m, steps, c.dt(0.05)) == resident


def test_bands_and_unpaired_sides_are_not_resident():
    c, m = model("sw", 3, 16, 16)
    m.SetBands(2)
    assert not gives_up(m, 5, c.dt(0.05))
    m.SetBands(0)
    assert gives_up(m, 5, c.dt(0.05))
    mesh = self_amd.Mesh2D.structured(6, 6, periodic=(True, True))
    mesh.sideInfo[0, 1, 2] = 9
    u = self_amd.ShallowWater(mesh, self_amd.SEMQuad(self_amd.Lagrange(3, self_amd.GAUSS, 3, self_amd.GAUSS), mesh))
    s = np.zeros(u.shape)
    s[:, 2] = 1.0
    u.SetSolution(s)
    assert not gives_up(u, 5, 1e-5)


@pytest.mark.parametrize("kind,N,nx,ny,metrics,hidden", [
    ("sw", 7, 10, 10, "affine", 0), ("sw", 3, 33, 31, "affine", 128), ("euler", 4, 9, 8, "nodal", 0)])
def test_every_reader_reports_it_and_a_new_state_ends_it(kind, N, nx, ny, metrics, hidden):
    c, m = model(kind, N, nx, ny, metrics, hidden)
    dt = c.dt(0.05)
    for _ in range(4):
        for st in range(3):
            m.Stage(st, dt)
    want = m.solution
    m.SetSolution(c.sol)
    assert gives_up(m, 4, dt)
    readers = [lambda: m.solution, m.CalculateTendency, m.flux_registers, lambda: m.Stage(0, dt),
               lambda: call("selfamd_model2d_synchronize", m._h), lambda: m.time_steps(3, dt)]
    if hidden:
        readers.append(m.closure_features)
    elif metrics == "affine":
        readers.append(lambda: self_amd.Batch([m], [dt]))
    for read in readers:
        with pytest.raises(SelfAmdError, match="gave up"):
            read()
    m._param(POLLS, 1 << 26)
    m.SetSolution(c.sol)
    m.ForwardStep(4, dt)
    np.testing.assert_array_equal(m.solution, want)


def test_scatter_into_a_model_ends_it():
    c, m = model("sw", 5, 9, 9, "affine")
    dt = c.dt(0.05)
    batch = self_amd.Batch([m], [dt])
    batch.ForwardStep(3)
    batch.scatter()
    want = m.solution
    m.ForwardStep(4, dt)
    later = m.solution
    assert gives_up(m, 4, dt)
    m._param(POLLS, 1 << 26)
    batch.scatter()
    np.testing.assert_array_equal(m.solution, want)
    m.ForwardStep(4, dt)
    np.testing.assert_array_equal(m.solution, later)
