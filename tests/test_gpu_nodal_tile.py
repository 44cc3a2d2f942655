"""The stage kernel's tile of nodal metrics at N = 5 (seven elements per block) against the oracle,
with one element, a block less one, a full block, and one more: the tendency and five steps."""
import numpy as np
import pytest

from tests.cases import Case, rel_err

import self_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["sw", "lsw", "euler"])
@pytest.mark.parametrize("nx,ny", [(1, 1), (6, 1), (7, 1), (4, 2), (5, 3)])
def test_partly_filled_blocks(kind, nx, ny):
    c = Case(kind, 5, nx, ny, bcid=self_amd.BC_NONORMALFLOW, metrics="nodal")
    m, _ = c.gpu_model()
    dt = c.dt(0.05)
    # the same FP64 sums in another order; a tendency is what is left of terms up to 1e4 times larger
    assert rel_err(m.CalculateTendency(), c.om.tendency()).max() <= 1e-11
    for _ in range(5):
        for st in range(3):
            m.Stage(st, dt)
    c.om.rk3_steps(5, dt)
    assert rel_err(m.solution, c.om.solution).max() <= 1e-12
    assert np.isfinite(m.solution).all()
