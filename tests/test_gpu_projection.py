"""The fine -> coarse L2 projection kernels against the FP64 oracle (oracle/closure.py) at the
edges of their ranges: the smallest sizes, chunks of sub-rows with a remainder, odd row
lengths, the longest run the LDS kernel takes, and the value-by-value path beyond it.

Tolerance: a result is a sum of r Pf products of factors along each direction; recursive
summation is off by at most (number of terms) u times the sum of magnitudes, which for these
factors (rows of Px sum to 1, their magnitudes to less than 4) is below 16 max|u|:
16 (2 r Pf) u with u = 2^-53, against the largest input."""
import numpy as np
import pytest

from oracle import closure as oc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nf,Nc,r,nxc,nyc,nvar", [
    (1, 1, 1, 1, 1, 1),     # the smallest
    (4, 2, 3, 3, 5, 1),     # odd rows, one variable
    (7, 3, 4, 9, 5, 3),     # all sub-rows at once
    (7, 4, 5, 3, 4, 4),     # two sub-rows at a time, one left over
    (15, 3, 6, 2, 2, 4),    # the longest run
    (3, 4, 2, 4, 3, 2),     # coarse degree above the fine one
    (4, 7, 2, 2, 3, 2),     # eight coarse nodes per direction: one sum per work-item
    (3, 3, 40, 1, 2, 3),    # beyond the kernel arguments: value by value
    (15, 1, 7, 2, 1, 4),    # beyond LDS: value by value
])
def test_projection_edges(Nf, Nc, r, nxc, nyc, nvar):
    import self_amd
    rng = np.random.default_rng(Nf + 10 * r + nvar)
    fine = rng.standard_normal((r * nxc * r * nyc, nvar, Nf + 1, Nf + 1))
    got = self_amd.project_l2_structured(fine, Nf, Nc, nxc, nyc, r, nvar).to_host()
    want = oc.project_l2_structured(fine, Nf, Nc, nxc, nyc, r)
    assert np.max(np.abs(got - want)) <= 16 * 2 * r * (Nf + 1) * 2.0 ** -53 * np.max(np.abs(fine))
