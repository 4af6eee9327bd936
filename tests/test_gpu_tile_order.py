"""Kernels whose workgroups take their tiles an eighth an XCD: every number of tiles modulo 8, fewer than 8 among them,
a last tile that is not full, and more workgroups than tiles (rows known on the device only are tested with whole nets).
Every row has to be written, once."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu

TILES = list(range(1, 18)) + [31, 40]


@pytest.mark.parametrize("C,ps", [(4, 9), (3, 4)])
def test_maxpool(scn, ctx, C, ps):
    rng = np.random.default_rng(C)
    inp = rng.standard_normal((300, C)).astype(np.float32)
    for tiles in TILES:
        n = 256 * tiles // (1 if C % 4 == 0 else C) - 2  # a lane has four channels, or one
        print("maxpool", C, n, flush=True)
        rules = rng.integers(0, 300, (n, ps)).astype(np.int32)
        out, choice = ctx.array(np.full((n, C), 7, np.float32)), ctx.empty((n, C), np.int32)
        ctx.maxpool(ctx.array(inp), out, ctx.array(rules), n, ps, C, choice)
        want, arg = orc.maxpool(inp, rules, n, ps, C)
        assert np.array_equal(out.download(), want) and np.array_equal(choice.download(), arg)
        d = ctx.array(np.zeros((300, C), np.float32))
        g = rng.integers(-4, 5, (n, C)).astype(np.float32)  # (whole numbers: their sums are exact in any order)
        ctx.maxpool_backward(d, ctx.array(g), n, C, choice)
        ref = np.zeros(300 * C)
        np.add.at(ref, arg.ravel(), g.ravel())
        assert np.array_equal(d.download().ravel(), ref.astype(np.float32))


# fused with the gather of 3 channels (128 rows a tile); split contraction (32 rows); tiles of 128 rows
@pytest.mark.parametrize("fs,nIn,N,rows,base", [(4, 3, 32, 128, 0), (4, 32, 32, 32, 0), (4, 32, 32, 128, 40000)])
def test_contractions(scn, ctx, fs, nIn, N, rows, base):
    rng = np.random.default_rng(fs * nIn)
    K = fs * nIn
    # (small whole numbers: products and sums are exact)
    inp, W = (rng.integers(-2, 3, s).astype(np.float32) for s in ((200, nIn), (K, N)))
    d_in, d_W, d_B = ctx.array(inp), ctx.array(W), ctx.array(np.zeros(N, np.float32))
    for tiles in TILES:
        n = base + rows * tiles - 3
        print("contraction", fs, nIn, N, n, flush=True)
        rules = rng.integers(0, 200, (n, fs)).astype(np.int32)
        out = ctx.array(np.full((n, N), 7, np.float32))
        ctx.conv_nin_forward(d_in, ctx.array(rules), fs, nIn, d_W, d_B, None, out, n, N, 1.0, scn.NOSIGMOID,
                             scn.FP32_PLANES)
        A = inp[rules].reshape(n, K)
        assert np.array_equal(out.download(), A @ W)
        if nIn == 32:
            dW = ctx.array(np.zeros((K, N), np.float32))
            g = rng.integers(-2, 3, (n, N)).astype(np.float32)
            ctx.sgemm_AtB(ctx.array(A), ctx.array(g), dW, n, K, N)
            assert np.array_equal(dW.download(), A.T @ g)
