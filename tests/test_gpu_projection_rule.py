"""The L2 projection on both sides of the line between its block-per-element and value-by-value
kernels, against the 64-bit oracle."""
import numpy as np
import pytest

from oracle import closure as oc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nf,Nc,r,nv,nxc,nyc", [
    (2, 2, 2, 1, 64, 62), (2, 2, 2, 1, 64, 63), (1, 1, 1, 3, 50, 40), (1, 1, 1, 3, 51, 40), (1, 3, 3, 2, 70, 60),
    (3, 3, 2, 3, 70, 60), (5, 6, 1, 1, 70, 60),
])
def test_projection_matches_oracle(Nf, Nc, r, nv, nxc, nyc):
    import self_amd
    fine = np.random.default_rng(Nf + nyc).standard_normal((r * nxc * r * nyc, nv, Nf + 1, Nf + 1))
    got = self_amd.project_l2_structured(fine, Nf, Nc, nxc, nyc, r, nv).to_host()
    want = oc.project_l2_structured(fine, Nf, Nc, nxc, nyc, r)
    assert np.max(np.abs(got - want)) <= 1e-14 * np.max(np.abs(want))
