"""Resident stepping with a closure attached (network, stage and mean mass correction of all stages
in one cooperative launch) against the same steps stage by stage, the network in its own launch:
the same bits, for every physics and degree it takes, hidden widths below, at and above one piece
of 64, single and partly filled row tiles, and a call after a call."""
import numpy as np
import pytest

import self_amd
from tests.cases import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,N,nx,ny,bc,hidden", [
    ("sw", 3, 64, 64, "periodic", 128), ("sw", 3, 5, 3, "wall", 128), ("sw", 3, 1, 1, "wall", 65), ("sw", 2, 9, 8, "periodic", 64),
    ("sw", 4, 33, 31, "wall", 100), ("sw", 1, 7, 6, "periodic", 17), ("lsw", 3, 17, 1, "open", 48), ("lsw", 4, 4, 4, "wall", 128),
    ("euler", 2, 13, 5, "wall", 80), ("euler", 3, 21, 20, "open", 128), ("euler", 4, 8, 6, "periodic", 64),
])
def test_resident_closure_equals_stages(kind, N, nx, ny, bc, hidden):
    bcid = self_amd.BC_NONORMALFLOW if bc == "wall" else self_amd.BC_RADIATION
    c = Case(kind, N, nx, ny, periodic=bc == "periodic", bcid=bcid, metrics="affine")
    m, _ = c.gpu_model()
    rng = np.random.default_rng(hidden)
    n_out = m.shape[1] * (N + 1) ** 2
    n_in = n_out + 3
    mlp = self_amd.MLP(n_in, hidden, n_out, nx * ny)
    w = lambda a, b: (rng.standard_normal((a, b)) / np.sqrt(a)).astype(np.float32)  # noqa: E731
    v = lambda a: (0.1 * rng.standard_normal(a)).astype(np.float32)  # noqa: E731
    mlp.set_params({"W1": w(n_in, hidden), "b1": v(hidden), "W2": w(hidden, hidden), "b2": v(hidden),
                    "W3": w(hidden, n_out), "b3": v(n_out)})
    m.SetClosure(mlp, 0.1 * v(n_in), 1 + v(n_in) ** 2, 1e-3 * v(n_out), np.full(n_out, 1e-2, np.float32))
    dt = c.dt(0.05)

    def run(step):
        m.SetSolution(c.sol)
        out = []
        for n in (4, 2, 1, 3):
            step(n)
            out.append(m.solution)
        return out

    def stages(n):
        for _ in range(n):
            for st in range(3):
                m.Stage(st, dt)

    want = run(stages)
    got = run(lambda n: m.ForwardStep(n, dt))
    for a, b in zip(got, want):
        assert np.isfinite(b).all()
        np.testing.assert_array_equal(a, b)
    # without the closure again: the ring serves the plain resident launch
    m.SetClosure(None)
    for a, b in zip(run(lambda n: m.ForwardStep(n, dt)), run(stages)):
        np.testing.assert_array_equal(a, b)
    assert np.abs(want[0] - m.solution).max() > 0
