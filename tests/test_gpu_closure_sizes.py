"""The closure's stage evaluation (features, network, correction, mean mass correction) at the sizes where
its launch changes: two 16-column tiles per wavefront (more than 128 hidden units), more row tiles than
a stage kernel adds up itself (512, beyond 8,192 elements), partly filled row tiles; against the 64-bit
oracles.

Tolerance: the network's FP32 sums, 4 u (sum of the reduction lengths) of the largest output (u = 2^-24),
scaled like the outputs, beside the rounding of two 64-bit tendencies."""
import numpy as np
import pytest

from oracle import closure as oc
from oracle import mlp as om

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


@pytest.mark.parametrize("N,nx,ny,hidden", [(3, 93, 89, 128), (3, 96, 97, 64), (3, 16, 15, 200), (3, 91, 93, 256), (2, 7, 5, 129),
                                            (5, 9, 7, 144)])
def test_stage_correction_matches_oracle(N, nx, ny, hidden):
    import self_amd
    from self_amd import workloads
    mesh = self_amd.Mesh2D.structured(nx, ny, periodic=(True, True))
    interp = self_amd.Lagrange(N, self_amd.GAUSS, N, self_amd.GAUSS)
    geom = self_amd.SEMQuad(interp, mesh)
    sol, topo = workloads.nonlinear_sw(geom.x.to_host(), interp.controlPoints, interp.qWeights, seed=1, width=0.3,
                                       vel_std=0.05)
    m = self_amd.ShallowWater(mesh, geom)
    m.SetTopography(topo)
    m.SetSolution(sol)
    J, d = geom.J.to_host()[:, 0, 0].copy(), geom.dsdx.to_host()
    n_out = 3 * (N + 1) ** 2
    n_in = n_out + 3
    rng = np.random.default_rng(hidden)
    net = self_amd.MLP(n_in, hidden, n_out, nx * ny)
    p32 = {k: v.astype(np.float32) for k, v in om.init_params(n_in, hidden, n_out, seed=2).items()}
    net.set_params(p32)
    norm = ((0.1 * rng.standard_normal(n_in)).astype(np.float32), (0.5 + rng.random(n_in)).astype(np.float32),
            (0.01 * rng.standard_normal(n_out)).astype(np.float32), (0.05 * (0.5 + rng.random(n_out))).astype(np.float32))
    plain = m.CalculateTendency()
    m.SetClosure(net, *norm)
    X = oc.features(sol, J, d[:, 0, 0, 0, 0].copy(), d[:, 0, 0, 1, 1].copy(), norm[0], norm[1])
    Y, _ = om.forward({k: v.astype(np.float64) for k, v in p32.items()}, X.astype(np.float64))
    want = oc.correction(Y, norm[2], norm[3], np.asarray(interp.qWeights), J, N, 3)
    got = m.CalculateTendency() - plain
    bound = 4 * U * (n_in + 2 * hidden + 16) * np.max(np.abs(Y)) * np.max(norm[3]) + 1e-14 * np.max(np.abs(plain))
    assert np.max(np.abs(got - want)) <= 2 * bound  # the correction and its mean
