"""First layers' matrices of columns in other than fours: the bits of the kernel for any shape (which takes outputs that do not
start on 16 bytes), and gathers of single words."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows: one over those of few, no whole workgroups'; columns below, at and above one workgroup's; 1 to 127 k
@pytest.mark.parametrize("M,K,N", [(513, 1, 4), (513, 9, 32), (1025, 27, 64), (2047, 27, 36), (5001, 54, 100), (777, 127, 160), (640, 81, 28),
                                   (4099, 2, 320)])
@pytest.mark.parametrize("act", ["RELU", "PRELU", "SOFTMAX", "TANH"])
def test_the_bits_of_the_general_kernel(scn, ctx, M, K, N, act):
    rng = np.random.default_rng(M + K)
    a = getattr(scn, act)
    A, W = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((K, N), dtype=np.float32)
    if K > 2:
        A[7, K - 1], A[M - 1, 0], A[9, 1] = np.inf, np.nan, -np.inf
    d_A, d_W = ctx.array(A), ctx.array(W)
    d_B, d_s = ctx.array(rng.standard_normal(N, dtype=np.float32)), ctx.array(rng.uniform(.1, .4, N).astype(np.float32))
    outs = [ctx.array(np.full(M * N + 200, 7, np.float32)) for _ in range(2)]
    for out, skew in zip(outs, (0, 1)):
        assert scn.lib().scn_nin_forward(ctx.h, d_A.ptr, d_W.ptr, d_B.ptr, d_s.ptr, out.ptr + 4 * skew, M, K, N, 0.5, a, scn.FP32) == 0
    x, y = (o.download() for o in outs)
    assert np.array_equal(x[:M * N], y[1:1 + M * N], equal_nan=True) and np.all(x[M * N:] == 7) and np.all(y[1 + M * N:] == 7)


@pytest.mark.parametrize("count", [1, 3, 4, 1023, 1027, 70001])
def test_gather_of_words(scn, ctx, count):
    rng = np.random.default_rng(count)
    x, rules = rng.standard_normal((91, 1), dtype=np.float32), rng.integers(-1, 91, count).astype(np.int32)
    out = ctx.array(np.full(count + 9, 7, np.float32))
    ctx.gather_rows(ctx.array(x), out, ctx.array(rules), count, 1)
    got = out.download()
    assert np.array_equal(got[:count], np.where(rules >= 0, x[np.maximum(rules, 0), 0], 0)) and np.all(got[count:] == 7)
