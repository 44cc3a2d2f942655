"""Device arrays that end before the call's data does are refused, as the copy calls refuse them, and
leave the state as it was; arrays that only a copy call can read are taken."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("missing", [1, 500])
def test_set_solution_refuses_a_short_device_array(missing):
    import self_amd
    mesh = self_amd.Mesh2D.structured(8, 8, periodic=(True, True))
    m = self_amd.ShallowWater(mesh, self_amd.SEMQuad(self_amd.Lagrange(3, self_amd.GAUSS, 3, self_amd.GAUSS), mesh))
    rng = np.random.default_rng(0)
    full = rng.random((64, 3, 4, 4)) + 1.0
    m.SetSolution(full)
    short = self_amd.DeviceArray.from_host(full.ravel()[:full.size - missing])
    with pytest.raises(self_amd.SelfAmdError):
        self_amd.call("selfamd_model2d_set_solution", m._h, short.ptr)
    assert np.array_equal(m.solution, full)
    # an array that ends with its allocation, and one inside a larger allocation
    m.SetSolution(2.0 * full)
    big = self_amd.DeviceArray.from_host(np.concatenate([np.zeros(6), full.ravel()]))
    self_amd.call("selfamd_model2d_set_solution", m._h, ctypes.c_void_p(big.ptr.value + 48))
    assert np.array_equal(m.solution, full)


@pytest.mark.parametrize("nH", [33, 257])  # row kernels, layer by layer
def test_mlp_backward_reads_its_cotangent_like_a_copy(nH):
    import self_amd
    from oracle import mlp as om
    rows, nIn, nOut = 70, 20, 17
    net = self_amd.MLP(nIn, nH, nOut, rows)
    net.set_params({k: v.astype(np.float32) for k, v in om.init_params(nIn, nH, nOut, seed=1).items()})
    rng = np.random.default_rng(nH)
    X = self_amd.DeviceArray.from_host(rng.standard_normal((rows, nIn)).astype(np.float32))
    dY = rng.standard_normal((rows, nOut)).astype(np.float32)
    dX = self_amd.DeviceArray((rows, nIn), np.float32)
    want_dX = net.backward(X, dY)
    want = net.get_grads()
    # host memory
    self_amd.call("selfamd_mlp_backward", net._h, X.ptr, ctypes.c_void_p(dY.ctypes.data), rows, 0, dX.ptr, None)
    assert (dX.to_host() == want_dX).all()
    assert all((net.get_grads()[k] == want[k]).all() for k in want)
    if nH > 256:
        return  # the runtime's own refusal would be the next call's last error
    # a device array that lacks the last row
    short = self_amd.DeviceArray.from_host(dY[:-1])
    with pytest.raises(self_amd.SelfAmdError):
        self_amd.call("selfamd_mlp_backward", net._h, X.ptr, short.ptr, rows, 0, dX.ptr, None)
