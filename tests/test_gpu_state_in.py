"""SetSolution from memory that a kernel on the model's device reads itself against memory that
needs a copy call first (not aligned to doubles): the same state, the same steps, for every physics, both
metric modes, degrees with full and with partly used blocks, and a last block that is not full."""
import ctypes

import numpy as np
import pytest

import self_amd
from self_amd._lib import call
from tests.cases import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,N,nx,ny,bc,metrics", [
    ("lsw", 1, 1, 1, "wall", "affine"), ("lsw", 7, 5, 1, "open", "affine"), ("sw", 2, 5, 7, "wall", "nodal"),
    ("sw", 3, 17, 1, "wall", "affine"), ("sw", 5, 3, 5, "periodic", "nodal"), ("euler", 4, 11, 1, "open", "affine"),
    ("euler", 6, 3, 2, "wall", "nodal"), ("euler", 7, 3, 3, "prescribed", "affine"),
])
def test_state_read_in_place_and_copied(kind, N, nx, ny, bc, metrics):
    ids = {"wall": self_amd.BC_NONORMALFLOW, "open": self_amd.BC_RADIATION, "prescribed": self_amd.BC_PRESCRIBED}
    c = Case(kind, N, nx, ny, periodic=bc == "periodic", bcid=ids.get(bc, self_amd.BC_NONORMALFLOW), metrics=metrics)
    dt = c.dt(0.05)
    data = np.ascontiguousarray(c.sol).view(np.uint8).reshape(-1)
    odd = self_amd.DeviceArray.from_host(np.concatenate([np.zeros(4, np.uint8), data, np.zeros(4, np.uint8)]))
    m, _ = c.gpu_model()
    runs = []
    for how in ("in place", "copied", "in place"):
        if how == "in place":
            m.SetSolution(c.sol)  # uploaded to a device array first
        else:
            call("selfamd_model2d_set_solution", m._h, ctypes.c_void_p(odd.ptr.value + 4))
        runs.append([m.solution])
        np.testing.assert_array_equal(runs[-1][0], c.sol)
        for n in (1, 3):
            m.ForwardStep(n, dt)
            runs[-1].append(m.solution)
        assert np.isfinite(runs[-1][-1]).all()
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            np.testing.assert_array_equal(a, b)
