"""The split contraction of more rows (k_nin_split64): the bits of the one of few rows, which takes the first rows by
themselves, whatever W comes as and whether the rows are gathered, and what fp32 makes of infinite operands."""
import numpy as np
import pytest

from test_gpu_capture import Graph

pytestmark = pytest.mark.gpu

# (rows, fs, nIn, N): as many workgroups as compute units and a few fewer, a row more or fewer than whole tiles; 14, 15, 27, 32
# and 80 blocks of 32 k, one to ten of them a wavefront; channels in 32s and in fours; columns that are no whole tile
SHAPES = [(16384, 14, 32, 64), (12383, 4, 120, 36), (8129, 24, 20, 100), (5440, 27, 32, 132), (2303, 4, 480, 448), (1216, 4, 640, 800),
          (8192, 1, 512, 128), (4033, 8, 128, 256)]


def inputs(ctx, rng, rows, fs, nIn, N):
    K = fs * nIn
    x = rng.standard_normal((900, nIn), dtype=np.float32)
    rules = rng.integers(-1, 900, (rows, fs)).astype(np.int32)
    W = (rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32)
    B = rng.uniform(-0.5, 0.5, N).astype(np.float32)
    return x, rules, W, B


@pytest.mark.parametrize("rows,fs,nIn,N", SHAPES)
@pytest.mark.parametrize("precision", ["FP32_PLANES", "BF16"])
def test_the_same_bits_as_few_rows(scn, ctx, rows, fs, nIn, N, precision):
    rng = np.random.default_rng(rows + N)
    p, K = getattr(scn, precision), fs * nIn
    if precision == "BF16":
        N, nIn = (N + 31) // 32 * 32, (nIn + 7) // 8 * 8
        rows = min(rows, 64 * (256 // -(-N // 64)))
        K = fs * nIn
        if K < 1024:
            pytest.skip("one plane: from 1024 k on")
        if not scn.lib().scn_conv_nin_supported_p(fs, nIn, N, p):
            pytest.skip("no fused kernel of this type")
    x, rules, W, B = inputs(ctx, rng, rows, fs, nIn, N)
    d_in, d_rules, d_W, d_B = (ctx.array(a) for a in (x, rules, W, B))
    d_slopes = ctx.array(rng.uniform(0.1, 0.4, N).astype(np.float32))
    size = -(-N // 32) * 32 * K * (6 if precision == "FP32_PLANES" else 2)
    assert scn.lib().scn_weight_image_bytes(ctx.h, rows, K, N, nIn, p) == (size if nIn % 32 == 0 else 0)
    image = ctx.empty((size // 4,), np.float32)
    ctx.weight_images_many([(d_W, image, K, N, 0, p)])
    outs = [ctx.array(np.full((rows + 64, N), 7, np.float32)) for _ in range(5)]
    matrix = ctx.empty((rows, K), np.float32)
    ctx.gather_rows(d_in, matrix, d_rules, rows * fs, nIn)
    print("split64", precision, rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, d_slopes, outs[0], rows, N, 1.0, scn.PRELU, p)
    ctx.conv_nin_forward_image(d_in, d_rules, fs, nIn, d_W, image, d_B, d_slopes, outs[1], rows, N, 1.0, scn.PRELU, p)
    ctx.conv_nin_forward_image(matrix, None, 1, K, d_W, image, d_B, d_slopes, outs[2], rows, N, 1.0, scn.PRELU, p)
    ctx.nin_forward(matrix, d_W, d_B, d_slopes, outs[3], rows, K, N, 1.0, scn.PRELU, p)
    with Graph(ctx) as g:
        ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, d_slopes, outs[4], rows, N, 1.0, scn.PRELU, p)
    g.replay(ctx)
    got = [o.download() for o in outs]
    g.close()
    few = 32 * (512 // -(-N // 32))  # two workgroups of 32 x 32 to a compute unit: few rows in either precision
    first = ctx.array(np.full((few + 64, N), 7, np.float32))
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, d_slopes, first, few, N, 1.0, scn.PRELU, p)
    first = first.download()
    assert few < rows and np.isfinite(first).all()
    for o in got:
        assert np.array_equal(o[:few], first[:few]) and np.array_equal(o, got[0]) and np.all(o[rows:] == 7)
    # (the rows behind those: the sums of their products, each rounded)
    a = np.where(rules[few:][:, :, None] >= 0, x[rules[few:]], 0).reshape(-1, K)
    w = W
    if precision == "BF16":
        def rounded(v):
            u = v.view(np.uint32).astype(np.uint64)
            return ((u + 0x7fff + (u >> 16 & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)
        a, w = rounded(np.ascontiguousarray(a, np.float32)), rounded(W)
    want = a.astype(np.float64) @ w.astype(np.float64) + B
    s = d_slopes.download()
    want = np.where(want > 0, want, want * s)
    bound = K * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64) + 1)
    assert np.all(np.abs(got[0][few:rows] - want) <= bound)


@pytest.mark.parametrize("M,K,N", [(8192, 512, 128), (12383, 448, 36), (2303, 1920, 448)])
def test_products_with_the_transpose(scn, ctx, M, K, N):
    rng = np.random.default_rng(M)
    D, Wt = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((N, K), dtype=np.float32)
    d_D, d_Wt, outs = ctx.array(D), ctx.array(Wt), [ctx.array(np.full((M + 64, N), 7, np.float32)) for _ in range(3)]
    workspace = ctx.empty((int(scn.lib().scn_sgemm_ABt_workspace(K, N)),), np.float32)
    print("split64 turned", M, K, N, flush=True)
    ctx.sgemm_ABt(d_D, d_Wt, outs[0], M, K, N, workspace)
    with Graph(ctx) as g:
        ctx.sgemm_ABt(d_D, d_Wt, outs[1], M, K, N, workspace)
    g.replay(ctx)
    ctx.nin_forward(d_D, ctx.array(np.ascontiguousarray(Wt.T)), ctx.array(np.zeros(N, np.float32)), None, outs[2], M, K, N, 1.0,
                    scn.NOSIGMOID, scn.FP32_PLANES)
    got = [o.download() for o in outs]
    g.close()
    assert all(np.array_equal(o, got[0]) and np.all(o[M:] == 7) for o in got)


@pytest.mark.parametrize("rows,fs,nIn,N", [(12383, 4, 120, 36), (1216, 4, 640, 800), (16384, 14, 32, 64)])
def test_infinite_operands_are_what_fp32_makes_of_them(scn, ctx, rows, fs, nIn, N):
    rng = np.random.default_rng(rows)
    special = np.array([np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 0], np.float32)
    x, rules, W, B = inputs(ctx, rng, rows, fs, nIn, N)
    W, K = W / 64, fs * nIn
    x[rng.choice(900, 12, False), rng.integers(0, nIn, 12)] = np.tile(special, 2)
    a = np.where(rules[:, :, None] >= 0, x[rules], 0).reshape(rows, K)
    some = np.unique(np.concatenate([np.arange(300), np.arange(rows - 300, rows)]))
    with np.errstate(invalid="ignore"):
        want = np.einsum("mk,kn->mn", a[some].astype(np.float64), W.astype(np.float64))
        scale = np.einsum("mk,kn->mn", np.abs(a[some]).astype(np.float64), np.abs(W).astype(np.float64))
    d_B, two = ctx.array(np.zeros(N, np.float32)), [ctx.array(np.full((rows, N), 7, np.float32)) for _ in range(2)]
    ctx.conv_nin_forward(ctx.array(x), ctx.array(rules), fs, nIn, ctx.array(W), d_B, None, two[0], rows, N, 1.0, scn.NOSIGMOID,
                         scn.FP32_PLANES)
    ctx.nin_forward(ctx.array(a), ctx.array(W), d_B, None, two[1], rows, K, N, 1.0, scn.NOSIGMOID, scn.FP32_PLANES)
    for out in two:
        got, sure = out.download()[some], np.isfinite(want)
        assert np.array_equal(got[~sure], want[~sure].astype(np.float32), equal_nan=True)
        assert np.all(np.abs(got[sure] - want[sure]) <= 2e-6 * scale[sure])
