"""A copy between device arrays has landed when it returns: a model's own stream, which does not
wait for the null stream, reads the copied values and not what the memory held before."""
import ctypes

import numpy as np
import pytest

import self_amd as sa
from self_amd._lib import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 160])
def test_copied_array_is_read_whole_by_a_model(n):
    mesh = sa.Mesh2D.structured(n, n)
    interp = sa.Lagrange(7, sa.GAUSS, 7, sa.GAUSS)
    m = sa.LinearShallowWater(mesh, sa.SEMQuad(interp, mesh), g=1.0)
    rng = np.random.default_rng(n)
    want = rng.standard_normal(m.shape)
    src = sa.DeviceArray.from_host(want)
    for _ in range(8):
        dst = sa.DeviceArray.from_host(np.full(m.shape, np.nan))
        call("selfamd_memcpy", dst.ptr, src.ptr, ctypes.c_size_t(src.nbytes), 3)
        m.SetSolution(dst)
        np.testing.assert_array_equal(m.solution, want)
