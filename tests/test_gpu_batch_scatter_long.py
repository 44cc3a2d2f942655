"""Scatter of arrays longer than one item of the copy list (2^18 doubles) beside short ones: whole items
and remainders, and more items than one launch takes."""
import numpy as np
import pytest

import self_amd
from tests.cases import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("runs", [[(7, 64, 64), (3, 5, 4), (7, 71, 67)], [(7, 160, 128)], [(5, 100, 91)] + [(3, 3, 3)] * 45])
def test_long_arrays_arrive_whole(runs):
    cases = [Case("sw", N, nx, ny, periodic=True, metrics="affine", seed=k) for k, (N, nx, ny) in enumerate(runs)]
    models = [c.gpu_model()[0] for c in cases]
    dt = 1e-5
    batch = self_amd.Batch(models, [dt] * len(models))
    batch.ForwardStep(1)
    batch.scatter()
    got = [m.solution for m in models]
    for m in models:
        m.ForwardStep(2, dt)
    later = [m.solution for m in models]
    for m, c, g, after in zip(models, cases, got, later):
        m.SetSolution(c.sol)
        m.ForwardStep(1, dt)
        np.testing.assert_array_equal(m.solution, g)
        m.ForwardStep(2, dt)  # state, RK register, traces and lagged velocities
        np.testing.assert_array_equal(m.solution, after)
