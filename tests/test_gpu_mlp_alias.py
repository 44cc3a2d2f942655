"""Network calls whose result lies over one of their operands, on the row kernels and layer by
layer, against the same calls on arrays of their own."""
import ctypes

import numpy as np
import pytest

from oracle import mlp as om

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _net(nIn, nH, nOut, rows, seed=3):
    import self_amd
    net = self_amd.MLP(nIn, nH, nOut, rows)
    net.set_params({k: v.astype(np.float32) for k, v in om.init_params(nIn, nH, nOut, seed=seed).items()})
    return net


def _at(array, floats):
    return ctypes.c_void_p(array.ptr.value + 4 * floats)


# hidden widths of one and two column tiles per wavefront, and beyond the row kernels; dX over X,
# over dY, and a few values into either
@pytest.mark.parametrize("nIn,nH,nOut,rows", [(20, 33, 20, 70), (51, 128, 48, 130), (30, 200, 17, 40), (12, 257, 12, 33)])
@pytest.mark.parametrize("over,shift", [("X", 0), ("dY", 0), ("X", 5), ("dY", 7)])
def test_backward_with_the_input_cotangent_over_an_operand(nIn, nH, nOut, rows, over, shift):
    import self_amd
    net = _net(nIn, nH, nOut, rows)
    rng = np.random.default_rng(nH + rows)
    X = rng.standard_normal((rows, nIn)).astype(np.float32)
    dY = rng.standard_normal((rows, nOut)).astype(np.float32)
    want_dX = net.backward(X, dY)
    want = net.get_grads()

    # one allocation: X, dY, and room for dX past the end of either
    room = rows * max(nIn, nOut) + shift
    mem = self_amd.DeviceArray((2 * room,), np.float32, zero=True)
    host = np.zeros(2 * room, np.float32)
    host[:X.size], host[room:room + dY.size] = X.ravel(), dY.ravel()
    mem.copy_from_host(host)
    at = shift if over == "X" else room + shift
    if over == "dY" and at + X.size > 2 * room:
        at = 2 * room - X.size
    self_amd.call("selfamd_mlp_backward", net._h, _at(mem, 0), _at(mem, room), rows, 0, _at(mem, at), None)
    got = net.get_grads()
    for k in want:  # the same kernels on the same values
        assert (got[k] == want[k]).all(), k
    # dX is a product of its own there: another order of nH FP32 terms
    dX = mem.to_host()[at:at + X.size].reshape(X.shape)
    assert np.max(np.abs(dX - want_dX)) <= 4 * U * (nH + 16) * np.max(np.abs(want_dX))


# outputs narrower, as wide and wider than the inputs: rows of Y over rows of X that other blocks read
@pytest.mark.parametrize("nIn,nH,nOut,rows", [(51, 128, 48, 4000), (20, 33, 20, 70), (17, 200, 60, 500), (12, 257, 9, 33)])
@pytest.mark.parametrize("shift", [0, 3])
def test_forward_over_its_input(nIn, nH, nOut, rows, shift):
    import self_amd
    net = _net(nIn, nH, nOut, rows)
    X = np.random.default_rng(rows).standard_normal((rows, nIn)).astype(np.float32)
    want = net.forward(X)
    mem = self_amd.DeviceArray((rows * max(nIn, nOut) + shift,), np.float32, zero=True)
    host = np.zeros(mem.shape, np.float32)
    host[:X.size] = X.ravel()
    mem.copy_from_host(host)
    self_amd.call("selfamd_mlp_forward", net._h, _at(mem, 0), _at(mem, shift), rows, None)
    got = mem.to_host()[shift:shift + want.size].reshape(want.shape)
    assert (got == want).all()


# narrow networks on both sides of the line from which the forward pass goes layer by layer
@pytest.mark.parametrize("nIn,nH,nOut,rows", [(3, 2, 4, 27903), (3, 2, 4, 27904), (17, 40, 5, 80128), (17, 40, 5, 80127)])
def test_narrow_networks_on_many_rows(nIn, nH, nOut, rows):
    import self_amd
    net = _net(nIn, nH, nOut, rows)
    rng = np.random.default_rng(rows)
    X = rng.standard_normal((rows, nIn)).astype(np.float32)
    p = {k: v.astype(np.float32).astype(np.float64) for k, v in om.init_params(nIn, nH, nOut, seed=3).items()}
    want, _ = om.forward(p, X.astype(np.float64))
    Xd = self_amd.DeviceArray.from_host(X)
    before = net.backward(Xd, want.astype(np.float32), want_dX=False), net.get_grads()
    got = net.forward(Xd)
    assert np.max(np.abs(got - want)) <= 4 * U * (nIn + 2 * nH + 16) * np.max(np.abs(want))
    # in place, and a backward pass after it
    mem = self_amd.DeviceArray((rows * max(nIn, nOut),), np.float32, zero=True)
    host = np.zeros(mem.shape, np.float32)
    host[:X.size] = X.ravel()
    mem.copy_from_host(host)
    self_amd.call("selfamd_mlp_forward", net._h, _at(mem, 0), _at(mem, 0), rows, None)
    assert (mem.to_host()[:want.size].reshape(want.shape) == got).all()
    net.backward(Xd, want.astype(np.float32), want_dX=False)
    after = net.get_grads()
    assert all((after[k] == before[1][k]).all() for k in after)
