"""Products with the transpose over no more than 32 columns of many rows: against 64-bit sums, not finite ones, captured."""
import numpy as np
import pytest

from test_gpu_capture import Graph

pytestmark = pytest.mark.gpu


# rows: the fewest, one more, no whole wavefronts' or workgroups'; columns: two tiles, one more, no fours, one to a workgroup
# and many; lengths of no whole step
@pytest.mark.parametrize("M,n,K", [(2048, 32, 64), (2049, 8, 65), (2111, 24, 100), (5003, 16, 897), (2305, 32, 4099), (30011, 32, 128),
                                   (131073, 32, 96)])
def test_products(scn, ctx, M, n, K):
    rng = np.random.default_rng(M)
    D, W = rng.standard_normal((M, n), dtype=np.float32), rng.standard_normal((K, n), dtype=np.float32)
    d_D, d_W, outs = ctx.array(D), ctx.array(W), [ctx.array(np.full((M + 300, K), 7, np.float32)) for _ in range(2)]
    workspace = ctx.empty((int(scn.lib().scn_sgemm_ABt_workspace(n, K)),), np.float32)
    print("narrow", M, n, K, flush=True)
    ctx.sgemm_ABt(d_D, d_W, outs[0], M, n, K, workspace)
    with Graph(ctx) as g:
        ctx.sgemm_ABt(d_D, d_W, outs[1], M, n, K, workspace)
    for _ in range(2):
        g.replay(ctx)
    a, b = (o.download() for o in outs)
    g.close()
    assert np.array_equal(a, b) and np.all(a[M:] == 7)
    some = np.unique(np.concatenate([np.arange(300), rng.integers(0, M, 2000), np.arange(M - 300, M)]))
    want, scale = D[some].astype(np.float64) @ W.astype(np.float64).T, np.abs(D[some]).astype(np.float64) @ np.abs(W).astype(np.float64).T
    # (each of n products and sums to half a unit of 2^-23 of no more than the scale)
    assert np.all(np.abs(a[some] - want) <= n * 2.0 ** -24 * scale)


def test_what_is_not_finite_is_what_fp32_makes_of_it(scn, ctx):
    rng = np.random.default_rng(1)
    M, n, K = 2200, 32, 200
    D, W = rng.standard_normal((M, n), dtype=np.float32), rng.standard_normal((K, n), dtype=np.float32)
    special = np.array([np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 0], np.float32)
    D[rng.choice(M, 12, False), rng.integers(0, n, 12)] = np.tile(special, 2)
    D[M - 1, 3], W[K - 1, 5], W[7, 0] = np.inf, -np.inf, np.nan
    out, workspace = ctx.array(np.full((M, K), 7, np.float32)), ctx.empty((int(scn.lib().scn_sgemm_ABt_workspace(n, K)),), np.float32)
    ctx.sgemm_ABt(ctx.array(D), ctx.array(W), out, M, n, K, workspace)
    with np.errstate(invalid="ignore", over="ignore"):
        want = np.einsum("mk,nk->mn", D.astype(np.float64), W.astype(np.float64))
        scale = np.einsum("mk,nk->mn", np.abs(D).astype(np.float64), np.abs(W).astype(np.float64))
    got = out.download()
    most = np.abs(want) > 3e38  # (a sum of that size may pass the largest float on the way, or be one)
    sure = np.isfinite(want) & ~most
    assert np.array_equal(got[~np.isfinite(want)], want[~np.isfinite(want)].astype(np.float32), equal_nan=True)
    assert np.all(np.abs(got[sure] - want[sure]) <= n * 2.0 ** -24 * scale[sure])


# (rows of few columns; by planes, in tiles and split; on the transpose)
@pytest.mark.parametrize("M,N,K,launches", [(3000, 32, 128, 1), (20000, 256, 128, 1), (500, 256, 128, 1), (90, 30, 20, 2), (3000, 20, 128, 2)])
def test_a_profile_has_no_spans_without_a_launch(scn, M, N, K, launches):
    rng = np.random.default_rng(M)
    c = scn.Context()
    D, W = c.array(rng.standard_normal((M, N), dtype=np.float32)), c.array(rng.standard_normal((K, N), dtype=np.float32))
    dA, ws = c.empty((M, K), np.float32), c.empty(scn.lib().scn_sgemm_ABt_workspace(N, K), np.float32)
    c.sgemm_ABt(D, W, dA, M, N, K, ws)
    c.prof_enable(True)
    c.sgemm_ABt(D, W, dA, M, N, K, ws)
    spans = c.prof_spans()
    c.prof_enable(False)
    print(spans, flush=True)
    assert len(spans) == launches
