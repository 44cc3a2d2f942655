"""The closure's adjoint, features to state cotangent in the network's launch, against FP64 numpy:
row tiles partly filled, full and past 16 rows, hidden widths of one and two tiles per wavefront
and off the multiples of four, and meshes with few and with many partial sums of the cotangent."""
import numpy as np
import pytest

import self_amd
from oracle import closure as oc
from oracle import mlp as om
from tests.test_gpu_closure import _coarse_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,N,hidden", [(2, 3, 128), (3, 2, 64), (4, 1, 30), (5, 4, 128), (17, 3, 200), (64, 3, 128),
                                        (40, 5, 17), (96, 3, 129)])
def test_closure_vjp_matches_fp64(n, N, hidden):
    m, S, J, d11, d22, qW = _coarse_model(n, N, seed=n)
    nOut = S[0].size
    nIn = nOut + 3
    rng = np.random.default_rng(100 * n + hidden)
    f32 = lambda a: np.asarray(a, np.float32)  # noqa: E731
    p = {k: f32(v + 0.05 * rng.standard_normal(v.shape)) for k, v in om.init_params(nIn, hidden, nOut, seed=n).items()}
    inMean, inScale = f32(0.1 * rng.standard_normal(nIn)), f32(0.5 + rng.random(nIn))
    outMean, outScale = f32(0.01 * rng.standard_normal(nOut)), f32(0.05 * (0.5 + rng.random(nOut)))
    net = self_amd.MLP(nIn, hidden, nOut, n * n)
    net.set_params(p)
    m.SetClosure(net, inMean, inScale, outMean, outScale)
    lam, mu0 = rng.standard_normal(S.shape), rng.standard_normal(S.shape)

    # FP64: cotangent of the outputs, through the network, to the parameters and the state
    q = {k: v.astype(np.float64) for k, v in p.items()}
    _, (X, z1, h1, z2, h2) = om.forward(q, oc.features(S, J, d11, d22, inMean, inScale).astype(np.float64))
    w = np.multiply.outer(qW, qW)
    omega = w[None] * J[:, None, None]
    dy = lam.copy()
    dy[:, 2] -= omega * (lam[:, 2].sum() / omega.sum())
    dy = dy.reshape(n * n, nOut) * outScale.astype(np.float64)
    dz2 = (dy @ q["W3"].T) * om.gelu_grad(z2)
    dz1 = (dz2 @ q["W2"].T) * om.gelu_grad(z1)
    mu = mu0 + ((dz1 @ q["W1"].T)[:, :nOut] / inScale[:nOut].astype(np.float64)).reshape(S.shape)
    # sums of at most max(hidden, rows per split) products in FP32, in any order: relative to the sum of
    # their magnitudes, terms * 2^-24 each layer; three layers
    terms = 3 * max(nIn, hidden, 144 if n > 64 else 128)
    a1, a2 = np.abs(dz1), np.abs(dz2)
    grads = {"W1": (X, dz1, a1), "W2": (h1, dz2, a2), "W3": (h2, dy, np.abs(dy))}
    net.zero_grads()
    for call in range(2):  # gradients add up over calls; a second call on the same model
        out = self_amd.DeviceArray.from_host(mu0)
        m.ClosureVJP(S, lam, out)
        assert np.abs(out.to_host() - mu).max() <= terms * 2.0 ** -24 * np.abs(mu - mu0).max() + 1e-14 * np.abs(mu).max()
        g = net.get_grads()
        for k, (a, d, ad) in grads.items():
            bound = 2 * (call + 1) * terms * 2.0 ** -24
            assert (np.abs(g[k] - (call + 1) * (a.T @ d)) <= bound * (np.abs(a).T @ ad).max()).all(), k
            assert (np.abs(g["b" + k[1]] - (call + 1) * d.sum(0)) <= bound * ad.sum(0).max()).all(), k
