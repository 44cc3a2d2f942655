"""The projection for every pair of fine and coarse degrees that has a kernel of its own, and the
ones beside them, against the oracle."""
import numpy as np
import pytest

from oracle import closure as oc

pytestmark = pytest.mark.gpu


# coarse degrees that the fine quadrature integrates
@pytest.mark.parametrize("Nf,Nc", [(f, c) for f in range(1, 9) for c in range(1, 7) if c <= 2 * f + 1])
def test_projection_degrees(Nf, Nc):
    import self_amd
    r, nvar = 1 + (Nf + Nc) % 3, 1 + (Nf * Nc) % 4
    fine = np.random.default_rng(10 * Nf + Nc).standard_normal((3 * r * 2 * r, nvar, Nf + 1, Nf + 1))
    got = self_amd.project_l2_structured(fine, Nf, Nc, 3, 2, r, nvar).to_host()
    want = oc.project_l2_structured(fine, Nf, Nc, 3, 2, r)
    # sums of (r (Nf + 1))^2 products; the factors of a sum over one direction add up to less than 16
    assert np.max(np.abs(got - want)) <= 16 * 2 * r * (Nf + 1) * 2.0 ** -53 * np.max(np.abs(fine))
