"""Device arrays that end before the call's data does are refused, as the copy calls refuse them, and
leave the state as it was."""
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
