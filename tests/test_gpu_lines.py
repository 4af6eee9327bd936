"""The contraction with both operands through LDS (rows by whole lines, weights from their image): the bits of the
kernels that convert the weights on the way, which a captured call takes, and nothing stored past the last row."""
import numpy as np
import pytest

from test_gpu_capture import Graph

pytestmark = pytest.mark.gpu

# (rows, fs, nIn, N): every tile of one and of three planes; a row more and fewer than whole groups of rows, columns that
# are no whole slice or tile, two, three and four blocks of 32 k (fewer than the ring holds), all filter positions
SHAPES = [(57251, 4, 32, 64), (28415, 4, 64, 96), (11393, 4, 96, 128), (6161, 4, 320, 100), (140033, 4, 96, 128),
          (16129, 2, 32, 36), (16385, 3, 32, 800), (9001, 8, 32, 800), (4160, 9, 32, 640), (40001, 27, 32, 60), (1025, 4, 640, 804)]


@pytest.mark.parametrize("rows,fs,nIn,N", SHAPES)
@pytest.mark.parametrize("precision", ["FP32_PLANES", "BF16"])
@pytest.mark.parametrize("gathered", [True, False])
def test_lines_give_the_same_bits(scn, ctx, rows, fs, nIn, N, precision, gathered):
    rng = np.random.default_rng(rows + N)
    K, nInRows, p = fs * nIn, 700, getattr(scn, precision)
    if precision == "BF16" and N % 32 != 0:
        N = (N + 31) // 32 * 32  # (what the fused kernels take)
    if gathered and not scn.lib().scn_conv_nin_supported_p(fs, nIn, N, p):
        pytest.skip("no fused kernel of this type")
    d_in = ctx.array(rng.standard_normal((nInRows, nIn), dtype=np.float32))
    d_rules = ctx.array(rng.integers(-1, nInRows, (rows, fs)).astype(np.int32))
    d_W = ctx.array((rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32))
    d_B = ctx.array(rng.uniform(-0.5, 0.5, N).astype(np.float32))
    d_slopes = ctx.array(rng.uniform(0.1, 0.4, N).astype(np.float32))
    one, two = (ctx.array(np.full((rows + 256, N), 7, np.float32)) for _ in range(2))
    matrix = None if gathered else ctx.empty((rows, K), np.float32)
    if not gathered:
        ctx.gather_rows(d_in, matrix, d_rules, rows * fs, nIn)

    def call(out):
        if gathered:
            ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, d_slopes, out, rows, N, 1.0, scn.PRELU, p)
        else:
            ctx.nin_forward(matrix, d_W, d_B, d_slopes, out, rows, K, N, 1.0, scn.PRELU, p)

    print("lines", precision, gathered, rows, fs, nIn, N, flush=True)
    call(one)
    ctx.sync()
    with Graph(ctx) as g:
        call(two)
    g.replay(ctx)
    ctx.sync()
    got, want = one.download(), two.download()
    g.close()
    assert np.all(got[rows:] == 7)
    assert np.isfinite(got).all() and np.array_equal(got, want)


@pytest.mark.parametrize("rows,fs,nIn,N", [(20011, 8, 64, 96), (40011, 8, 64, 96), (70145, 9, 64, 128), (33025, 8, 32, 64), (9001, 8, 160, 256)])
def test_bf16_rows(scn, ctx, rows, fs, nIn, N):
    rng = np.random.default_rng(rows)
    K = fs * nIn
    d_in, d_in16 = ctx.array(rng.standard_normal((900, nIn), dtype=np.float32)), ctx.empty((900, nIn), np.float32)
    d_rules = ctx.array(rng.integers(-1, 900, (rows, fs)).astype(np.int32))
    d_W, d_B = ctx.array((0.1 * rng.standard_normal((K, N))).astype(np.float32)), ctx.array(np.zeros(N, np.float32))
    one, two = (ctx.array(np.full((rows + 256, N), 7, np.float32)) for _ in range(2))
    print("lines of bf16 rows", rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward_a16(d_in, 900, d_in16, d_rules, fs, nIn, d_W, d_B, None, one, rows, N, 1.0, scn.RELU)
    with Graph(ctx) as g:
        ctx.conv_nin_forward_a16(d_in, 900, d_in16, d_rules, fs, nIn, d_W, d_B, None, two, rows, N, 1.0, scn.RELU)
    g.replay(ctx)
    got, want = one.download(), two.download()
    g.close()
    assert np.all(got[rows:] == 7) and np.array_equal(got, want)


@pytest.mark.parametrize("rows,fs,nIn,N", [(28415, 4, 64, 96), (9001, 8, 32, 36), (33001, 2, 64, 160), (20001, 27, 32, 64)])
@pytest.mark.parametrize("precision", ["FP32_PLANES", "BF16"])
def test_weights_laid_out_ahead(scn, ctx, rows, fs, nIn, N, precision):
    """several layers' in one launch, as they stand and as the filters of the layer they are turned from"""
    rng = np.random.default_rng(rows)
    K, p = fs * nIn, getattr(scn, precision)
    N = (N + 31) // 32 * 32 if precision == "BF16" else N
    d_in = ctx.array(rng.standard_normal((500, nIn), dtype=np.float32))
    d_rules = ctx.array(rng.integers(-1, 500, (rows, fs)).astype(np.int32))
    W = (rng.standard_normal((fs, nIn, N)) * 0.1).astype(np.float32)
    d_W, d_turned = ctx.array(W.reshape(K, N)), ctx.array(np.ascontiguousarray(W.transpose(0, 2, 1)).reshape(fs * N, nIn))
    d_B = ctx.array(rng.uniform(-0.5, 0.5, N).astype(np.float32))
    size = (N + 31) // 32 * 32 * K * (6 if precision == "FP32_PLANES" else 2)
    # (the wider of these shapes are faster with their weights converted on the way)
    assert scn.lib().scn_weight_image_bytes(ctx.h, rows, K, N, nIn, p) in (0, size)
    assert scn.lib().scn_weight_image_bytes(ctx.h, 28415, 256, 96, 64, p) == 96 * 256 * (6 if precision == "FP32_PLANES" else 2)
    assert scn.lib().scn_weight_image_bytes(ctx.h, 32, K, N, nIn, p) == 0  # (the split contraction: W as it stands)
    images = [ctx.empty((size // 4,), np.float32) for _ in range(3)]
    print("images", precision, rows, fs, nIn, N, flush=True)
    ctx.weight_images_many([(d_W, images[0], K, N, 0, p), (d_turned, images[1], K, N, fs, p), (d_W, images[2], K, N, 0, p)])
    outs = [ctx.array(np.full((rows, N), 7, np.float32)) for _ in range(4)]
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, None, outs[3], rows, N, 1.0, scn.RELU, p)
    for image, out in zip(images, outs):
        ctx.conv_nin_forward_image(d_in, d_rules, fs, nIn, d_W, image, d_B, None, out, rows, N, 1.0, scn.RELU, p)
    want = outs[3].download()
    for out in outs[:3]:
        assert np.array_equal(out.download(), want)
    matrix, plain = ctx.empty((rows, K), np.float32), ctx.array(np.full((rows, N), 7, np.float32))
    ctx.gather_rows(d_in, matrix, d_rules, rows * fs, nIn)
    ctx.conv_nin_forward_image(matrix, None, 1, K, d_W, images[0], d_B, None, plain, rows, N, 1.0, scn.RELU, p)
    assert np.array_equal(plain.download(), want)


def test_a_matrix_of_more_columns_than_there_are_numbers_is_refused(scn, ctx):
    buf = ctx.empty((64, 64), np.float32)
    for fs, nIn in ((1 << 16, (1 << 16) + 1), (1 << 30, 4), (0, 32), (4, 0)):
        with pytest.raises(scn.ScnError):  # (without rows: nothing is launched either way)
            ctx.conv_nin_forward_image(buf, None, fs, nIn, buf, None, buf, None, buf, 0, 64, 1.0, scn.RELU, scn.FP32_PLANES)


def test_no_image_of_more_columns_than_the_stores_reach(scn, ctx):
    """64 rows of the output in a gigabyte"""
    for p in (scn.FP32_PLANES, scn.BF16):
        assert scn.lib().scn_weight_image_bytes(ctx.h, 10000, 64, 1 << 22, 64, p) > 0
        assert scn.lib().scn_weight_image_bytes(ctx.h, 10000, 64, (1 << 22) + 32, 64, p) == 0


@pytest.mark.parametrize("M,N,K", [(4001, 64, 96), (33333, 128, 384), (9000, 96, 512)])
def test_products_with_the_transpose(scn, ctx, M, N, K):
    rng = np.random.default_rng(M)
    D, W = rng.standard_normal((M, N), dtype=np.float32), rng.standard_normal((K, N), dtype=np.float32)
    out, workspace = ctx.array(np.full((M + 256, K), 7, np.float32)), ctx.empty(N * K + K, np.float32)
    print("lines ABt", M, N, K, flush=True)
    ctx.sgemm_ABt(ctx.array(D), ctx.array(W), out, M, N, K, workspace)
    got = out.download()
    want = D.astype(np.float64) @ W.T.astype(np.float64)
    scale = np.abs(D).astype(np.float64) @ np.abs(W.T).astype(np.float64)
    assert np.all(got[M:] == 7)
    # products to 2^-25, one rounding of the sum every few k (as in test_gpu_planes.py)
    assert (np.abs(got[:M] - want) / scale).max() <= 2e-6


# rows: part of a step of sixteen, a step and a row more, fewer steps than the ring holds, several ranges of rows;
# columns that are no whole tile, two filter positions to a tile of 64 (or, in fours, three)
@pytest.mark.parametrize("M", [1, 15, 17, 129, 391, 2051, 40003])
@pytest.mark.parametrize("fs,nIn,N", [(3, 36, 44), (4, 32, 64), (2, 96, 160), (9, 8, 4)])
def test_weight_gradients_by_lines(scn, ctx, M, fs, nIn, N):
    rng = np.random.default_rng(M + nIn)
    K = fs * nIn
    x, D = rng.standard_normal((300, nIn), dtype=np.float32), rng.standard_normal((M, N), dtype=np.float32)
    rules = rng.integers(-1, 300, (M, fs)).astype(np.int32)
    pitch = (M + 15) // 16 * 16
    positions = ctx.array(np.ascontiguousarray(np.pad(rules.T, ((0, 0), (0, pitch - M)), constant_values=-1)))
    dense = np.where(rules[:, :, None] >= 0, x[np.maximum(rules, 0)], 0).reshape(M, K).astype(np.float32)
    want, scale = dense.T.astype(np.float64) @ D, np.abs(dense.T).astype(np.float64) @ np.abs(D) + 1e-30
    d_x, d_D, d_A = ctx.array(x), ctx.array(D), ctx.array(dense)
    dW, dB, plain = ctx.array(np.full((K, N), 7, np.float32)), ctx.array(np.full(N, 7, np.float32)), ctx.empty((K, N), np.float32)
    print("dW by lines", M, fs, nIn, N, flush=True)
    ctx.conv_AtB(d_x, positions, fs, nIn, d_D, dW, M, N, d_db=dB)
    ctx.sgemm_AtB(d_A, d_D, plain, M, K, N)
    # products to 2^-25 and one rounding of a sum every few rows, as in test_gpu_planes.py
    for got in (dW, plain):
        assert (np.abs(got.download() - want) / scale).max() <= 2e-6
    assert (np.abs(dB.download() - D.sum(0, dtype=np.float64)) / (np.abs(D).sum(0) + 1e-30)).max() <= 2e-6


# plain rows of which a compute unit has several tiles (k_nin_lines' LONG): two blocks of k, which a tile's requests are ahead
# of its last block by, and more; slices of columns that do not divide an XCD's workgroups (640, 1280: 5 and 10); the last tile
# of one row, of all but one; rows that are not finite in the first, a middle and the last tile, which are taken again there
@pytest.mark.parametrize("M,K,N", [(128 * 300 + 1, 64, 384), (128 * 523 - 1, 128, 128), (256 * 300 + 77, 64, 64), (33001, 128, 256),
                                   (70003, 128, 96), (40000, 96, 640), (20011, 320, 1280), (50001, 256, 192), (35001, 384, 112),
                                   (50001, 96, 160)])
def test_several_tiles_to_a_workgroup(scn, ctx, M, K, N):
    rng = np.random.default_rng(M + K + N)
    A, W = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((N, K), dtype=np.float32)
    odd = [0, M // 2, M - 1]
    A[odd, 3] = [np.inf, np.nan, -np.inf]
    print("several tiles", M, K, N, flush=True)
    out, ws = ctx.array(np.full((M, N), 7, np.float32)), ctx.empty(int(scn.lib().scn_sgemm_ABt_workspace(K, N)), np.float32)
    ctx.sgemm_ABt(ctx.array(A), ctx.array(W), out, M, K, N, ws)
    got = out.download()
    with np.errstate(invalid="ignore"):
        assert np.array_equal(got[odd], A[odd, 3:4] * W[:, 3], equal_nan=True)
    A[odd] = 0
    got[odd] = 0
    for r in range(0, M, 20000):
        a = A[r:r + 20000].astype(np.float64)
        assert np.all(np.abs(got[r:r + 20000] - a @ W.T.astype(np.float64)) <= 2e-6 * (np.abs(a) @ np.abs(W.T).astype(np.float64)))


# the same forward, with bias and activation, in every tile that is launched so (test_planes_choice.py: these reach all), the bits
# of the kernels that convert the weights on the way; two, three and more blocks of k, the last of them rows and results that
# are more than the caches
SEVERAL = [(38401, 64, 384), (40000, 96, 640), (33001, 64, 160), (200003, 96, 64), (33001, 128, 256), (33001, 512, 256),
           (35001, 384, 112), (33001, 512, 128), (720001, 64, 32)]


@pytest.mark.parametrize("M,K,N", SEVERAL)
@pytest.mark.parametrize("act", ["LEAKYRELU", "PRELU"])
def test_several_tiles_to_a_workgroup_forward(scn, ctx, M, K, N, act):
    rng = np.random.default_rng(M + K + N)
    A, W = rng.standard_normal((M, K), dtype=np.float32), (rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32)
    A[[0, M // 2, M - 1], 3] = [np.inf, np.nan, -np.inf]  # (taken again, in the first, a middle and the last tile)
    d_A, d_W, d_B = ctx.array(A), ctx.array(W), ctx.array(rng.uniform(-0.5, 0.5, N).astype(np.float32))
    slopes = ctx.array(rng.uniform(0.1, 0.4, N).astype(np.float32)) if act == "PRELU" else None
    image = ctx.empty(((N + 31) // 32 * 32 * K * 6 // 4,), np.float32)
    ctx.weight_images_many([(d_W, image, K, N, 0, scn.FP32_PLANES)])
    one, two = (ctx.array(np.full((M + 256, N), 7, np.float32)) for _ in range(2))
    print("several tiles forward", M, K, N, act, flush=True)
    ctx.conv_nin_forward_image(d_A, None, 1, K, d_W, image, d_B, slopes, one, M, N, 1.0, getattr(scn, act), scn.FP32_PLANES)
    ctx.sync()
    with Graph(ctx) as g:
        ctx.nin_forward(d_A, d_W, d_B, slopes, two, M, K, N, 1.0, getattr(scn, act), scn.FP32_PLANES)
    g.replay(ctx)
    ctx.sync()
    got, want = one.download(), two.download()
    g.close()
    assert np.all(got[M:] == 7) and np.array_equal(got, want, equal_nan=True)
