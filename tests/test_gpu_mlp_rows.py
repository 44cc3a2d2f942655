"""The closure network's matrix-core row kernels at the edges of their tiles (16 rows, 16
columns, 64 reduction indices, one or two column tiles per wavefront, 32 x 32 gradient tiles)
and the layer-by-layer path beyond their range, against the FP64 oracle (oracle/mlp.py).

Tolerance: a dot product of K FP32 terms that round independently is off by about
sqrt(K) u sum|terms| / sqrt(K) = u sum|terms|, and for terms of random sign sum|terms| is about
sqrt(K) times the result's typical size; against the largest result, with the layers' errors
adding up, 4 u (sum of the reduction lengths of a path) bounds it with room (u = 2^-24)."""
import numpy as np
import pytest

from oracle import mlp as om

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
SHAPES = [
    (51, 128, 48, 17),    # the configured network, one row into a second tile
    (1, 1, 1, 1),         # the smallest
    (16, 16, 16, 16),     # one tile of everything
    (17, 33, 15, 15),     # just over and under a tile; unaligned weight rows
    (64, 128, 64, 128),   # exact pieces
    (65, 129, 5, 129),    # a second column tile per wavefront; a second row split
    (30, 200, 27, 300),   # second tile in some wavefronts only; unaligned output rows
    (243, 256, 75, 65),   # the widest hidden layers of the row kernels
    (8, 257, 6, 40),      # beyond them: layer by layer
    (9, 20, 257, 33),     # more outputs than the row kernels take: layer by layer
]


@pytest.mark.parametrize("nIn,nH,nOut,rows", SHAPES)
def test_row_kernels_match_oracle(nIn, nH, nOut, rows):
    import self_amd
    rng = np.random.default_rng(nIn + 7 * nH + rows)
    p32 = {k: (v + (0.1 * rng.standard_normal(v.shape) if k.startswith("b") else 0)).astype(np.float32)
           for k, v in om.init_params(nIn, nH, nOut, seed=rows).items()}
    p = {k: v.astype(np.float64) for k, v in p32.items()}
    net = self_amd.MLP(nIn, nH, nOut, rows + 3)
    net.set_params(p32)
    X = (1.5 * rng.standard_normal((rows, nIn))).astype(np.float32)
    T = rng.standard_normal((rows, nOut)).astype(np.float32)
    Xd, Td = self_amd.DeviceArray.from_host(X), self_amd.DeviceArray.from_host(T)

    def check(got, want, length, what):
        err = np.max(np.abs(got - want)) / np.max(np.abs(want))
        assert err <= 4 * U * length, (what, err, 4 * U * length)

    forward, back = nIn + 2 * nH + 16, nIn + 4 * nH + nOut + rows + 16
    y, _ = om.forward(p, X.astype(np.float64))
    check(net.forward(X), y, forward, "forward")

    loss, want = om.loss_and_grads(p, X.astype(np.float64), T.astype(np.float64))
    got_loss = net.loss_grad(Xd, Td)
    assert abs(got_loss - loss) <= 4 * U * back * loss
    grads = net.get_grads()
    for k in want:
        check(grads[k], want[k], back, k)

    # the same cotangent given from outside, gradients added to what is there, and the input cotangent
    dY = (2.0 * (y - T) / y.size).astype(np.float32)
    dX = net.backward(X, dY, accumulate=True)
    twice = net.get_grads()
    for k in want:
        check(twice[k], 2.0 * want[k], back, k)
    dz2 = (dY.astype(np.float64) @ p["W3"].T)
    z1 = X.astype(np.float64) @ p["W1"] + p["b1"]
    z2 = om.gelu(z1) @ p["W2"] + p["b2"]
    check(dX, ((dz2 * om.gelu_grad(z2)) @ p["W2"].T * om.gelu_grad(z1)) @ p["W1"].T, back, "dX")
    # deterministic
    net.loss_grad(Xd, Td)
    assert all(np.array_equal(net.get_grads()[k], grads[k]) for k in grads)
