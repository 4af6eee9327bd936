"""Long contractions captured into a HIP graph.  The context's copy of a layer's weights belongs to the context's own
calls: a graph, which may be replayed beside them, converts the weights on the way and gives the same bits."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Graph:
    """what the calls inside `with` queue on a context's stream (the HIP runtime the library itself is linked to)"""

    def __init__(self, ctx):
        self.hip, self.stream = C.CDLL("libamdhip64.so"), C.c_void_p(ctx.stream())
        self.graph, self.exe = C.c_void_p(), C.c_void_p()

    def __enter__(self):
        # (global mode: an allocation during the capture would be an error)
        assert self.hip.hipStreamBeginCapture(self.stream, 0) == 0
        return self

    def __exit__(self, *_):
        assert self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph)) == 0
        n = C.c_size_t()
        assert self.hip.hipGraphGetNodes(self.graph, None, C.byref(n)) == 0
        self.nodes = n.value
        assert self.hip.hipGraphInstantiate(C.byref(self.exe), self.graph, None, None, 0) == 0

    def replay(self, ctx):
        assert self.hip.hipGraphLaunch(self.exe, C.c_void_p(ctx.stream())) == 0

    def close(self):
        self.hip.hipGraphExecDestroy(self.exe)
        self.hip.hipGraphDestroy(self.graph)


# conv: fp32 in three planes, bf16 in one; product with W^T.  All long enough for the context's copy of the weights.
@pytest.mark.parametrize("what,kernels", [("FP32_PLANES", 1), ("BF16", 1), ("ABt", 2)])
def test_a_graph_keeps_off_the_contexts_weights(scn, what, kernels):
    rng = np.random.default_rng(3)
    M, fs, nIn, N = 66000, 27, 64, 64
    K = fs * nIn
    ctx, side = scn.Context(0), scn.Context(0)
    if what == "ABt":  # [M x 256] times the transpose of [512 x 256]
        D = ctx.array(rng.standard_normal((M, 256), dtype=np.float32))
        Ws = [ctx.array(rng.standard_normal((512, 256), dtype=np.float32)) for _ in range(2)]
        workspaces = [ctx.empty(scn.lib().scn_sgemm_ABt_workspace(256, 512), np.float32) for _ in range(2)]
        outs = [ctx.array(np.full((M, 512), 7, np.float32)) for _ in range(4)]

        def call(i, out):
            ctx.sgemm_ABt(D, Ws[i], outs[out], M, 256, 512, workspaces[i])
    else:
        x, rules = ctx.array(rng.standard_normal((500, nIn), dtype=np.float32)), ctx.array(
            rng.integers(-1, 500, (M, fs)).astype(np.int32))
        Ws = [ctx.array((rng.standard_normal((K, N)) * 0.05).astype(np.float32)) for _ in range(2)]
        B = ctx.array(np.zeros(N, np.float32))
        outs = [ctx.array(np.full((M, N), 7, np.float32)) for _ in range(4)]

        def call(i, out):
            ctx.conv_nin_forward(x, rules, fs, nIn, Ws[i], B, None, outs[out], M, N, 1.0, scn.RELU, getattr(scn, what))

    print("capture", what, flush=True)
    call(0, 0)
    call(1, 1)
    ctx.sync()
    want = [outs[0].download(), outs[1].download()]
    assert np.isfinite(want[0]).all() and not np.array_equal(*want)
    with Graph(ctx) as g:
        call(0, 2)
    # no copy of the weights in it: the contraction alone, or with the caller's own transposition
    assert g.nodes == kernels
    for _ in range(4):  # on another stream, beside calls of the context with other weights
        outs[2].upload(np.full_like(want[0], 7))
        outs[3].upload(np.full_like(want[1], 7))
        g.replay(side)
        call(1, 3)
        side.sync()
        ctx.sync()
        assert np.array_equal(outs[2].download(), want[0]) and np.array_equal(outs[3].download(), want[1])
    g.close()
    side.close()
    for a in outs + Ws:
        a.free()
    ctx.close()
