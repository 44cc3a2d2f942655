"""Operator kernels over all instantiated degrees (P = 2 .. 8), the runtime-P path beyond them,
slab counts that do not fill the last block, and arrays that are not 16-byte aligned, against
the oracle.

Tolerance: both sides add the same at most 2 P + 4 products, so they differ by at most the
rounding of each step, (2 P + 6) u of the sum of magnitudes, bounded here by the largest
product (max|M| max|f|) times the number of terms; copies must be equal."""
import ctypes

import numpy as np
import pytest

import oracle
import self_amd
from self_amd import _lib

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


def call(name, *args):
    _lib.call(name, *[a.ptr if isinstance(a, self_amd.DeviceArray) else a for a in args], None)
    self_amd.synchronize()


@pytest.mark.parametrize("nEl,nVar", [(1, 1), (11, 3)])
@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7, 8, 11])
def test_operator_sizes(N, nEl, nVar):
    rng = np.random.default_rng(100 * N + nVar)
    P = N + 1
    L = oracle.lagrange_init(N, oracle.GAUSS, N, oracle.GAUSS)
    D = self_amd.DeviceArray.from_host
    terms = 2 * P + 6

    def check(got, want, scale, what):
        err = np.abs(got - want).max()
        assert err <= terms * U * terms * scale, (what, N, err)

    bM, mb = D(L["bMatrix"]), np.abs(L["bMatrix"]).max()
    for ncomp, name in ((1, "scalar"), (2, "vector"), (4, "tensor")):
        tail = {1: (), 2: (2,), 4: (2, 2)}[ncomp]
        f = rng.normal(size=(nEl, nVar, P, P) + tail)
        out = self_amd.DeviceArray((nEl, 4, nVar, P) + tail)
        call(f"selfamd_{name}_boundary_interp_2d", bM, D(f), out, N, nVar, nEl)
        want = getattr(oracle, f"{name}_boundary_interp")(N, L["bMatrix"], f)
        check(out.to_host(), want, mb * np.abs(f).max(), name)
    f = rng.normal(size=(nEl, nVar, P, P, 2))
    bF = rng.normal(size=(nEl, 4, nVar, P))
    out = self_amd.DeviceArray((nEl, nVar, P, P))
    call("selfamd_vector_divergence_2d", D(L["dMatrix"]), D(f), out, N, nVar, nEl)
    check(out.to_host(), oracle.vector_divergence(N, L["dMatrix"], f), np.abs(L["dMatrix"]).max() * np.abs(f).max(), "strong")
    call("selfamd_vector_dg_divergence_2d", D(L["dgMatrix"]), bM, D(L["qWeights"]), D(f), D(bF), out, N, nVar, nEl)
    scale = max(np.abs(L["dgMatrix"]).max() * np.abs(f).max(), mb * np.abs(bF).max() / L["qWeights"].min())
    check(out.to_host(), oracle.vector_dg_divergence(N, L["dgMatrix"], L["bMatrix"], L["qWeights"], f, bF), scale, "weak")

    # streaming updates: aligned, and one value past an aligned address
    n = nEl * nVar * P * P
    G, S, d = (rng.normal(size=n + 1) for _ in range(3))
    for off in (0, 1):
        Gd, Sd, dd, out = D(G), D(S), D(d), self_amd.DeviceArray((n + 1,))
        at = [ctypes.c_void_p(x.ptr.value + 8 * off) for x in (Gd, Sd, dd, out)]
        call("selfamd_calculate_dsdt", at[0], at[1], at[3], N, nVar, nEl)
        np.testing.assert_array_equal(out.to_host()[off:off + n], S[off:off + n] - G[off:off + n])
        call("selfamd_update_grk", at[0], at[1], at[2], -5.0 / 9.0, 15.0 / 16.0, 1e-3, N, nVar, nEl)
        g = -5.0 / 9.0 * G[off:off + n] + d[off:off + n]
        np.testing.assert_array_equal(Gd.to_host()[off:off + n], g)
        np.testing.assert_array_equal(Sd.to_host()[off:off + n], S[off:off + n] + (15.0 / 16.0 * 1e-3) * g)
        rest = slice(n, n + 1) if off == 0 else slice(0, 1)
        np.testing.assert_array_equal(Gd.to_host()[rest], G[rest])


@pytest.mark.parametrize("N", [1, 4, 6, 8])
def test_exchange_and_pointwise_sizes(N):
    rng = np.random.default_rng(N)
    P, nVar = N + 1, 3
    mesh = self_amd.Mesh2D.structured(3, 5, periodic=(True, False))
    nEl = mesh.nElem
    D = self_amd.DeviceArray.from_host
    si = self_amd.DeviceArray.from_host(mesh.sideInfo)
    b = rng.normal(size=(nEl, 4, nVar, P))
    ext = self_amd.DeviceArray(b.shape, zero=True)
    call("selfamd_side_exchange_scalar_2d", D(b), ext, si, N, nVar, nEl)
    np.testing.assert_array_equal(ext.to_host(), oracle.side_exchange_scalar(N, mesh.sideInfo, b))
    J = 0.5 + rng.random((nEl, P, P))
    f = rng.normal(size=(nEl, nVar, P, P))
    fd = D(f)
    call("selfamd_jacobian_weight_2d", D(J), fd, N, nVar, nEl)
    np.testing.assert_array_equal(fd.to_host(), f / J[:, None])
    dsdx = rng.normal(size=(nEl, P, P, 2, 2))
    fv = rng.normal(size=(nEl, nVar, P, P, 2))
    fvd = D(fv)
    call("selfamd_contravariant_projection_2d", D(dsdx), fvd, N, nVar, nEl)
    d = dsdx.reshape(nEl, 1, P, P, 4)
    want = np.stack((d[..., 0] * fv[..., 0] + d[..., 1] * fv[..., 1], d[..., 2] * fv[..., 0] + d[..., 3] * fv[..., 1]), -1)
    np.testing.assert_array_equal(fvd.to_host(), want)
    # node-wise physics against closed forms
    sol = np.stack((rng.normal(size=(nEl, P, P)), rng.normal(size=(nEl, P, P)), 1.0 + rng.random((nEl, P, P))), 1)
    vel = sol[:, :2] / sol[:, 2:]
    flux = self_amd.DeviceArray((nEl, 3, P, P, 2))
    call("selfamd_sw2d_flux", flux, D(sol), D(np.moveaxis(vel, 1, -1)[:, None]), ctypes.c_double(9.81), N, nEl)
    p = 0.5 * 9.81 * sol[:, 2] * sol[:, 2]
    want = np.stack((np.stack((vel[:, 0] * sol[:, 0] + p, vel[:, 1] * sol[:, 0]), -1),
                     np.stack((vel[:, 0] * sol[:, 1], vel[:, 1] * sol[:, 1] + p), -1),
                     np.stack((sol[:, 0], sol[:, 1]), -1)), 1)
    np.testing.assert_allclose(flux.to_host(), want, rtol=8 * U, atol=8 * U * np.abs(want).max())
