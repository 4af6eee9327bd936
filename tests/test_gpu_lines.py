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
