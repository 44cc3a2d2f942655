"""Resident stepping over calls of more launches and more waits than one: each wait is bounded by
itself, so a call may be as long as it likes."""
import numpy as np
import pytest

import self_amd
from tests.cases import Case

pytestmark = pytest.mark.gpu


def test_long_call_equals_short_calls():
    """1.2 million stages of six blocks, each of which waits for its neighbours in every stage."""
    c = Case("lsw", 7, 3, 2, bcid=self_amd.BC_NONORMALFLOW, metrics="affine")
    m, _ = c.gpu_model()
    dt = c.dt(0.01)
    m.ForwardStep(400_000, dt)
    long = m.solution
    m.SetSolution(c.sol)
    for _ in range(100):
        m.ForwardStep(4000, dt)
    assert np.isfinite(long).all()
    np.testing.assert_array_equal(m.solution, long)
