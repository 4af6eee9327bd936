"""Small contractions of plain rows in planes, and those of one tile of columns; SCN_FP32 stays on the fp32 MFMA."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# plain rows below and above four tiles of 32 x 32 to a compute unit, SCN_FP32_PLANES alone
SMALL = [(9307, 2, 32, 64), (5461, 4, 64, 96), (10924, 4, 64, 96), (9307, 8, 12, 96), (6561, 4, 96, 160), (300, 2, 32, 36)]


@pytest.mark.parametrize("rows,fs,nIn,N", SMALL)
def test_small_plain_contractions_without_an_image(scn, ctx, rows, fs, nIn, N):
    """converted on the way, from an image made by the call or made before, through rules: the same bits"""
    rng = np.random.default_rng(rows + N)
    K, p = fs * nIn, scn.FP32_PLANES
    d_in = ctx.array(rng.standard_normal((900, nIn), dtype=np.float32))
    d_rules = ctx.array(rng.integers(-1, 900, (rows, fs)).astype(np.int32))
    d_W = ctx.array((rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32))
    d_B = ctx.array(rng.uniform(0.1, 0.4, N).astype(np.float32))
    matrix, image = ctx.empty((rows, K), np.float32), ctx.empty((-(-N // 32) * 32 * K * 6 // 4,), np.float32)
    ctx.gather_rows(d_in, matrix, d_rules, rows * fs, nIn)
    ctx.weight_images_many([(d_W, image, K, N, 0, p)])
    outs = [ctx.array(np.full((rows + 128, N), 7, np.float32)) for _ in range(3)]
    print("small plain", rows, fs, nIn, N, flush=True)
    ctx.nin_forward(matrix, d_W, d_B, None, outs[0], rows, K, N, 1.0, scn.RELU, p)
    ctx.conv_nin_forward_image(matrix, None, 1, K, d_W, image, d_B, None, outs[1], rows, N, 1.0, scn.RELU, p)
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, None, outs[2], rows, N, 1.0, scn.RELU, p)
    got = [o.download() for o in outs]
    assert all(np.array_equal(o, got[0]) and np.all(o[rows:] == 7) for o in got)


@pytest.mark.parametrize("rows,K,N", [(78124, 800, 32), (90000, 768, 32), (30000, 96, 20), (61000, 512, 64), (90000, 512, 128)])
def test_shorter_contractions_stay_on_the_fp32_mfma(scn, ctx, rows, K, N):
    """fused and not the same bits, not the planes'; products with the transpose, in planes, of 128 x 32 a workgroup"""
    rng = np.random.default_rng(rows)
    A, W = rng.standard_normal((rows, K), dtype=np.float32), (rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)
    d_A, d_W, d_B = ctx.array(A), ctx.array(W), ctx.array(np.zeros(N, np.float32))
    each = ctx.array(np.arange(rows, dtype=np.int32))
    outs = [ctx.array(np.full((rows + 128, N), 7, np.float32)) for _ in range(4)]
    ctx.nin_forward(d_A, d_W, d_B, None, outs[0], rows, K, N, 1.0, scn.NOSIGMOID, scn.FP32)
    ctx.conv_nin_forward(d_A, each, 1, K, d_W, d_B, None, outs[1], rows, N, 1.0, scn.NOSIGMOID, scn.FP32)
    ctx.nin_forward(d_A, d_W, d_B, None, outs[2], rows, K, N, 1.0, scn.NOSIGMOID, scn.FP32_PLANES)
    ctx.sgemm_ABt(d_A, ctx.array(np.ascontiguousarray(W.T)), outs[3], rows, K, N,
                  ctx.empty((int(scn.lib().scn_sgemm_ABt_workspace(K, N)),), np.float32))
    got = [o.download() for o in outs]
    assert all(np.all(o[rows:] == 7) for o in got)
    assert np.array_equal(got[0], got[1]) and not np.array_equal(got[0], got[2]) and np.array_equal(got[2], got[3])
    want = A.astype(np.float64) @ W.astype(np.float64)
    error = [np.linalg.norm(o[:rows] - want) / np.linalg.norm(want) for o in got]
    assert error[2] < error[0] < 2e-6
