"""Network calls on a stream under capture: the graph's replays, with eager work between them, give what
the calls give."""
import ctypes

import numpy as np
import pytest

from oracle import mlp as om

pytestmark = pytest.mark.gpu


def _hip():
    import self_amd
    self_amd.load()
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64.so" in line)
    return ctypes.CDLL(path)


# row kernels, narrow layers (forward), layer by layer; mode 0: global capture, 2: relaxed
@pytest.mark.parametrize("nIn,nH,nOut,rows", [(51, 128, 48, 300), (3, 2, 4, 30000), (12, 257, 9, 64)])
@pytest.mark.parametrize("mode", [0, 2])
def test_captured_calls_replay(nIn, nH, nOut, rows, mode):
    import self_amd
    hip = _hip()

    def ok(status):
        assert status == 0, status

    net = self_amd.MLP(nIn, nH, nOut, rows)
    net.set_params({k: v.astype(np.float32) for k, v in om.init_params(nIn, nH, nOut, seed=5).items()})
    rng = np.random.default_rng(rows)
    inputs = [(rng.standard_normal((rows, nIn)).astype(np.float32), rng.standard_normal((rows, nOut)).astype(np.float32))
              for _ in range(3)]
    X, dY = (self_amd.DeviceArray.from_host(a) for a in inputs[0])
    Y, dX = self_amd.DeviceArray((rows, nOut), np.float32), self_amd.DeviceArray((rows, nIn), np.float32)
    stream, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    ok(hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1))
    ok(hip.hipStreamBeginCapture(stream, mode))
    self_amd.call("selfamd_mlp_forward", net._h, X.ptr, Y.ptr, rows, stream)
    self_amd.call("selfamd_mlp_backward", net._h, X.ptr, dY.ptr, rows, 0, dX.ptr, stream)
    ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)))
    ok(hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, 0))
    try:
        for x, d in inputs + inputs[:1]:
            want_Y, want_dX = net.forward(x), net.backward(x, d)
            want = net.get_grads()
            X.copy_from_host(x)
            dY.copy_from_host(d)
            ok(hip.hipGraphLaunch(run, stream))
            ok(hip.hipStreamSynchronize(stream))
            assert (Y.to_host() == want_Y).all() and (dX.to_host() == want_dX).all()
            got = net.get_grads()
            assert all((got[k] == want[k]).all() for k in want)
    finally:
        hip.hipGraphExecDestroy(run)
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(stream)
