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


# fused with the gather of 3 channels (32 rows a tile, and 64 from 49153 rows on); split contraction (32 rows); tiles of
# no more than 128 rows
@pytest.mark.parametrize("fs,nIn,N,rows,base", [(4, 3, 32, 32, 0), (4, 3, 32, 64, 49152), (4, 32, 32, 32, 0),
                                                (4, 32, 32, 128, 40000)])
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


# k_nin_lines (there is an image for it), whose tiles have 64, 128 or 256 rows: in steps of 64, so that all remainders
# come up for each; one slice of columns, several, and columns to an XCD where the image is the larger part
@pytest.mark.parametrize("precision", ["FP32_PLANES", "BF16"])
@pytest.mark.parametrize("fs,nIn,N,base,gathered", [(4, 64, 96, 28000, True), (4, 320, 480, 6000, True), (2, 64, 64, 9000, False),
                                                    (4, 640, 832, 1100, False)])
def test_lines(scn, ctx, precision, fs, nIn, N, base, gathered):
    rng = np.random.default_rng(N)
    K, p = fs * nIn, getattr(scn, precision)
    inp, W = (rng.integers(-2, 3, s).astype(np.float32) for s in ((200, nIn), (K, N)))
    d_in, d_W, d_B = ctx.array(inp), ctx.array(W), ctx.array(np.zeros(N, np.float32))
    image = ctx.empty(K * N * 6 // 4, np.float32)
    ctx.weight_images_many([(d_W, image, K, N, 0, p)])
    every = rng.integers(0, 200, (base + 64 * 40, fs)).astype(np.int32)
    A = inp[every].reshape(-1, K)
    want = A @ W
    rows = [base + 64 * tiles - 3 for tiles in range(1, 41)]
    # (the cost may prefer another kernel for some of them: the same bits)
    assert sum(scn.lib().scn_weight_image_bytes(ctx.h, n, K, N, nIn if gathered else K, p) > 0 for n in rows) >= 32
    for n in rows:
        print("lines", precision, fs, nIn, N, n, flush=True)
        out = ctx.array(np.full((n + 64, N), 7, np.float32))
        if gathered:
            ctx.conv_nin_forward_image(d_in, ctx.array(every[:n]), fs, nIn, d_W, image, d_B, None, out, n, N, 1.0, scn.NOSIGMOID, p)
        else:
            ctx.conv_nin_forward_image(ctx.array(A[:n]), None, 1, K, d_W, image, d_B, None, out, n, N, 1.0, scn.NOSIGMOID, p)
        got = out.download()
        assert np.array_equal(got[:n], want[:n]) and np.all(got[n:] == 7)


# of bf16 rows: tiles of 128 rows by 128 columns, or by 64
@pytest.mark.parametrize("fs,nIn,N,base", [(8, 160, 256, 9000), (8, 32, 64, 33000)])
def test_lines_of_bf16_rows(scn, ctx, fs, nIn, N, base):
    rng = np.random.default_rng(N)
    K = fs * nIn
    inp, W = (rng.integers(-2, 3, s).astype(np.float32) for s in ((200, nIn), (K, N)))
    d_in, d_W, d_B, d_in16 = ctx.array(inp), ctx.array(W), ctx.array(np.zeros(N, np.float32)), ctx.empty((200, nIn), np.float32)
    every = rng.integers(0, 200, (base + 128 * 16, fs)).astype(np.int32)
    want = inp[every].reshape(-1, K) @ W
    for tiles in range(1, 17):
        n = base + 128 * tiles - 3
        print("lines of bf16 rows", fs, nIn, N, n, flush=True)
        out = ctx.array(np.full((n + 64, N), 7, np.float32))
        ctx.conv_nin_forward_a16(d_in, 200, d_in16, ctx.array(every[:n]), fs, nIn, d_W, d_B, None, out, n, N, 1.0, scn.NOSIGMOID)
        got = out.download()
        assert np.array_equal(got[:n], want[:n]) and np.all(got[n:] == 7)
