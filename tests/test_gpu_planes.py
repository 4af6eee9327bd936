"""The contraction on bf16 planes (SCN_FP32_PLANES, and SCN_FP32 where it goes there): every tile, the split
contraction, the image of W, ragged rows and columns, fused with the gather and not."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


# (rows, fs, nIn, N): split contraction from one row on, N no multiple of a tile; every tile converted on the way,
# a block more or less than a full group of rows; an odd number of blocks; channels looked up in fours; images
@pytest.mark.parametrize("rows,fs,nIn,N", [(1, 4, 32, 32), (33, 3, 32, 100), (257, 9, 96, 36), (300, 4, 24, 64),
                                           (20000, 4, 32, 64), (40001, 4, 32, 32), (66049, 3, 32, 96), (30000, 8, 12, 64),
                                           (70001, 4, 64, 128), (65537, 27, 64, 64), (33005, 9, 96, 96)])
@pytest.mark.parametrize("act", ["RELU", "PRELU"])
def test_planes_against_float64(scn, ctx, rows, fs, nIn, N, act):
    a = getattr(scn, act)
    rng = np.random.default_rng(rows + fs + nIn + N)
    nInRows, K = 500, fs * nIn
    inp = (rng.standard_normal((nInRows, nIn)) * 10.0 ** rng.uniform(-3, 3, (nInRows, 1))).astype(np.float32)
    rules = rng.integers(0, nInRows, (rows, fs)).astype(np.int32)
    rules[rng.random((rows, fs)) < 0.1] = -1
    W = (rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32)
    B = rng.uniform(-0.5, 0.5, N).astype(np.float32)
    pr = rng.uniform(0.1, 0.4, N).astype(np.float32)
    d_in, d_rules, d_W, d_B, d_pr = (ctx.array(x) for x in (inp, rules, W, B, pr))
    fused, two = ctx.array(np.full((rows, N), 7, np.float32)), ctx.array(np.full((rows, N), 7, np.float32))
    print("planes", rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, d_pr, fused, rows, N, 1.0, a, scn.FP32_PLANES)
    g = ctx.empty((rows, K), np.float32)
    ctx.gather_rows(d_in, g, d_rules, rows * fs, nIn)
    ctx.nin_forward(g, d_W, d_B, d_pr, two, rows, K, N, 1.0, a, scn.FP32_PLANES)
    got = fused.download()
    assert np.array_equal(got, two.download())
    some = np.unique(np.concatenate([np.arange(min(rows, 300)), np.arange(max(0, rows - 300), rows)]))
    A = np.where(rules[some, :, None] >= 0, inp[np.maximum(rules[some], 0)], 0).reshape(len(some), K).astype(np.float32)
    want = orc.nin_forward(A, W, B, pr, 1.0, a, f64=True)
    scale = np.abs(A).astype(np.float64) @ np.abs(W).astype(np.float64) + np.abs(B)
    err = np.abs(got[some] - want) / scale
    # products to 2^-25, one rounding of the sum every few k: within the plain fp32 accumulation's own error
    plain = np.abs(orc.nin_forward(A, W, B, pr, 1.0, a) - want) / scale
    assert err.max() <= 2e-6 and np.sqrt((err ** 2).mean()) <= np.sqrt((plain ** 2).mean()) + 1e-8


# rows gathered, W streamed from its image: whole and broken groups of rows, an odd and an even number of blocks, columns
# that are no whole slice
@pytest.mark.parametrize("rows,fs,nIn,N", [(70144, 9, 64, 128), (70145, 27, 32, 128), (65791, 27, 64, 64), (40001, 27, 96, 160),
                                           (33024, 12, 160, 224)])
@pytest.mark.parametrize("a16", [False, True])
def test_streamed_weights_give_the_same_bits(scn, ctx, rows, fs, nIn, N, a16):
    rng = np.random.default_rng(rows + fs)
    d_in = ctx.array(rng.standard_normal((900, nIn), dtype=np.float32))
    d_rules = ctx.array(rng.integers(-1, 900, (rows, fs)).astype(np.int32))
    d_W = ctx.array(rng.standard_normal((fs * nIn, N), dtype=np.float32))
    d_B = ctx.array(rng.uniform(-0.5, 0.5, N).astype(np.float32))
    one, two = (ctx.array(np.full((rows, N), 7, np.float32)) for _ in range(2))
    print("streamed", rows, fs, nIn, N, a16, flush=True)
    if a16:
        ctx.conv_nin_forward_a16(d_in, 900, ctx.empty((900, nIn), np.float32), d_rules, fs, nIn, d_W, d_B, None, one, rows, N,
                                 1.0, scn.RELU)
    else:
        ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, None, one, rows, N, 1.0, scn.RELU, scn.FP32_PLANES)
    g = ctx.empty((rows, fs * nIn), np.float32)
    ctx.gather_rows(d_in, g, d_rules, rows * fs, nIn)
    ctx.nin_forward(g, d_W, d_B, None, two, rows, fs * nIn, N, 1.0, scn.RELU, scn.BF16 if a16 else scn.FP32_PLANES)
    assert np.array_equal(one.download(), two.download())


def test_fp32_takes_the_planes_where_they_pay(scn, ctx):
    """few rows and long contractions: the same bits as SCN_FP32_PLANES"""
    rng = np.random.default_rng(5)
    for M, K, N in ((100, 256, 64), (200000, 1728, 64)):
        A = ctx.array(rng.standard_normal((M, K), dtype=np.float32))
        W = ctx.array(rng.standard_normal((K, N), dtype=np.float32))
        B = ctx.array(np.zeros(N, np.float32))
        out = [ctx.empty((M, N), np.float32) for _ in range(2)]
        for o, precision in zip(out, (scn.FP32, scn.FP32_PLANES)):
            ctx.nin_forward(A, W, B, None, o, M, K, N, 1.0, scn.NOSIGMOID, precision)
        assert np.array_equal(out[0].download(), out[1].download())


# split contraction; tiles converted on the way, in fours, from the image
@pytest.mark.parametrize("rows,fs,nIn,N", [(40, 4, 32, 36), (20000, 4, 32, 64), (30000, 8, 12, 64), (70001, 4, 64, 128),
                                           (65537, 9, 64, 64)])
def test_infinite_operands_are_what_fp32_makes_of_them(scn, ctx, rows, fs, nIn, N):
    """infinities, NaN and values past the largest bf16 in few rows of A: no NaN where the sum has none"""
    rng = np.random.default_rng(rows + N)
    K, special = fs * nIn, np.array([np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 0], np.float32)
    inp = rng.standard_normal((600, nIn)).astype(np.float32)
    inp[rng.choice(600, 12, False), rng.integers(0, nIn, 12)] = np.tile(special, 2)
    rules = rng.integers(0, 600, (rows, fs)).astype(np.int32)
    W = (0.5 * rng.standard_normal((K, N)) / K).astype(np.float32)
    A = inp[rules].reshape(rows, K)
    some = np.unique(np.concatenate([np.arange(min(rows, 300)), np.arange(max(0, rows - 300), rows)]))
    with np.errstate(invalid="ignore"):
        want = np.einsum("mk,kn->mn", A[some].astype(np.float64), W.astype(np.float64))
        scale = np.einsum("mk,kn->mn", np.abs(A[some]).astype(np.float64), np.abs(W).astype(np.float64))
    d_rules, d_in, d_W, d_B = ctx.array(rules), ctx.array(inp), ctx.array(W), ctx.array(np.zeros(N, np.float32))
    d_A, fused, two, dA = ctx.array(A), *(ctx.array(np.full((rows, N), 7, np.float32)) for _ in range(3))
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, None, fused, rows, N, 1.0, scn.NOSIGMOID, scn.FP32_PLANES)
    ctx.nin_forward(d_A, d_W, d_B, None, two, rows, K, N, 1.0, scn.NOSIGMOID, scn.FP32_PLANES)
    ctx.sgemm_ABt(d_A, ctx.array(np.ascontiguousarray(W.T)), dA, rows, K, N, ctx.empty(N * K + K, np.float32))
    for name, out in (("fused", fused), ("two", two), ("ABt", dA)):
        got, sure = out.download()[some], np.isfinite(want)
        assert np.array_equal(got[~sure], want[~sure].astype(np.float32), equal_nan=True), name
        assert np.all(np.abs(got[sure] - want[sure]) <= 2e-6 * scale[sure]), name
    # dW = A^T D over the first rows, an infinity in a row of its own and in D
    M = min(rows, 2000)
    A = rng.standard_normal((M, K), dtype=np.float32)
    D = (0.1 * rng.standard_normal((M, N)) / M).astype(np.float32)
    A[3, 5], A[M - 1, 7], A[4, 9], D[M // 2, 11] = np.inf, -np.inf, 3.4e38, np.inf
    dW = ctx.array(np.zeros((K, N), np.float32))
    ctx.sgemm_AtB(ctx.array(A), ctx.array(D), dW, M, K, N)
    with np.errstate(invalid="ignore"):
        want, got = np.einsum("mk,mn->kn", A.astype(np.float64), D.astype(np.float64)), dW.download()
    scale = np.einsum("mk,mn->kn", np.abs(A).astype(np.float64), np.abs(D).astype(np.float64))
    sure = np.isfinite(want)
    assert np.array_equal(got[~sure], want[~sure].astype(np.float32), equal_nan=True)
    assert np.all(np.abs(got[sure] - want[sure]) <= 2e-6 * scale[sure])


# one row; fewer rows than a step; odd K or N (no pairs of columns); every tile; ragged row ranges
@pytest.mark.parametrize("M,K,N", [(1, 32, 32), (15, 12, 32), (129, 27, 33), (130, 34, 31), (1000, 66, 100),
                                   (40001, 12, 32), (30011, 256, 96), (5000, 128, 62), (70003, 432, 128)])
def test_weight_gradient_and_input_gradient(scn, ctx, M, K, N):
    rng = np.random.default_rng(M + K + N)
    A, D = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((M, N), dtype=np.float32)
    W, start = rng.standard_normal((K, N), dtype=np.float32), rng.standard_normal((K, N), dtype=np.float32)
    dW = ctx.array(start)
    print("products", M, K, N, flush=True)
    ctx.sgemm_AtB(ctx.array(A), ctx.array(D), dW, M, K, N, accumulate=True)
    scale = np.abs(A).astype(np.float64).T @ np.abs(D).astype(np.float64) + np.abs(start)
    assert np.all(np.abs(dW.download() - start - A.astype(np.float64).T @ D) <= 2e-6 * scale)
    dA = ctx.array(np.full((M, K), 7, np.float32))
    ctx.sgemm_ABt(ctx.array(D), ctx.array(W), dA, M, N, K, ctx.empty(N * K + K, np.float32))
    some = np.unique(np.concatenate([np.arange(min(M, 300)), np.arange(max(0, M - 300), M)]))
    scale = np.abs(D[some]).astype(np.float64) @ np.abs(W).astype(np.float64).T
    assert np.all(np.abs(dA.download()[some] - D[some].astype(np.float64) @ W.astype(np.float64).T) <= 2e-6 * scale)


@pytest.mark.parametrize("M,N", [(1, 1), (3, 4), (700, 260), (5001, 64), (9000, 37), (40000, 96)])
@pytest.mark.parametrize("act", ["RELU", "PRELU"])
def test_activation_backward_column_sums(scn, ctx, M, N, act):
    rng = np.random.default_rng(M + N)
    out, delta = (rng.standard_normal((M, N)).astype(np.float32) for _ in range(2))
    pr = rng.uniform(0.1, 0.4, N).astype(np.float32)
    d, db, dp = ctx.array(delta), ctx.array(np.zeros(N, np.float32)), ctx.array(np.zeros(N, np.float32))
    ctx.activation_backward(ctx.array(out), d, M, N, getattr(scn, act), ctx.array(pr), db, dp)
    want = np.where(out > 0, delta, delta * pr if act == "PRELU" else np.float32(0)).astype(np.float32)
    assert np.array_equal(d.download(), want)
    assert np.allclose(db.download(), want.astype(np.float64).sum(0), atol=2e-6 * M ** 0.5 * 4 + 1e-6, rtol=1e-5)
    if act == "PRELU":
        slope = np.where(out > 0, 0, delta * (out / pr)).astype(np.float64).sum(0)
        assert np.allclose(dp.download(), slope, atol=1e-5 * M ** 0.5 * 4 + 1e-5, rtol=1e-4)


# one plane, up to four column tiles a wavefront: N a multiple of them or not, ragged rows, few and many blocks; bf16
# rows and fp32 rows; a window of channels in other than 32s
@pytest.mark.parametrize("rows,fs,nIn,N", [(12801, 4, 64, 128), (33005, 9, 96, 160), (20001, 27, 32, 96), (9001, 4, 160, 320),
                                           (6001, 4, 480, 640), (60001, 8, 24, 224)])
def test_one_plane_against_float64(scn, ctx, rows, fs, nIn, N):
    rng = np.random.default_rng(rows + N)
    K = fs * nIn
    inp = rng.standard_normal((700, nIn), dtype=np.float32)
    rules = rng.integers(-1, 700, (rows, fs)).astype(np.int32)
    W = (rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32)
    B = rng.uniform(-0.5, 0.5, N).astype(np.float32)
    d_in, d_rules, d_W, d_B = (ctx.array(x) for x in (inp, rules, W, B))
    one, two, three = (ctx.array(np.full((rows, N), 7, np.float32)) for _ in range(3))
    print("one plane", rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, None, one, rows, N, 1.0, scn.RELU, scn.BF16)
    ctx.conv_nin_forward_a16(d_in, 700, ctx.empty((700, nIn), np.float32), d_rules, fs, nIn, d_W, d_B, None, two, rows, N,
                             1.0, scn.RELU)
    g = ctx.empty((rows, K), np.float32)
    ctx.gather_rows(d_in, g, d_rules, rows * fs, nIn)
    ctx.nin_forward(g, d_W, d_B, None, three, rows, K, N, 1.0, scn.RELU, scn.BF16)
    got = one.download()
    assert np.array_equal(got, two.download()) and np.array_equal(got, three.download())

    def bf16(x):
        u = x.view(np.uint32)
        return ((u + 0x7fff + (u >> 16 & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)

    some = np.unique(np.concatenate([np.arange(300), np.arange(rows - 300, rows)]))
    A = np.where(rules[some, :, None] >= 0, inp[np.maximum(rules[some], 0)], 0).reshape(len(some), K).astype(np.float32)
    want = orc.nin_forward(bf16(A), bf16(W), B, None, 1.0, scn.RELU, f64=True)
    scale = np.abs(A).astype(np.float64) @ np.abs(W).astype(np.float64) + np.abs(B)
    # products exact, their sum in fp32: a rounding every eight or sixteen of the K
    assert np.all(np.abs(got[some] - want) <= 2e-6 * scale)


# a contraction of the tiles, the split contraction, the input gradient, the weight gradient
@pytest.mark.parametrize("what,M,K,N", [("forward", 40000, 1728, 64), ("forward", 4000, 1728, 64), ("ABt", 40000, 256, 512),
                                        ("AtB", 40000, 256, 96)])
def test_a_net_that_diverged_costs_a_few_times_what_a_sound_one_does(scn, ctx, what, M, K, N):
    """weights that have all gone to NaN, or to infinities (which leave no early way out): sums that are not finite are
    taken again a tile at a time"""
    import time
    rng = np.random.default_rng(M + K)
    A = ctx.array(rng.standard_normal((M, K), dtype=np.float32))
    D = ctx.array(rng.standard_normal((M, N), dtype=np.float32))
    B, out, ws = ctx.array(np.zeros(N, np.float32)), ctx.empty((M, N), np.float32), ctx.empty(N * K + N, np.float32)
    dW, best = ctx.array(np.zeros((K, N), np.float32)), {}
    W = rng.standard_normal((K, N), dtype=np.float32)
    for name, value in (("sound", None), ("nan", np.nan), ("inf", np.inf)):
        w = W if value is None else np.where(W > 0, np.float32(value), -np.float32(value))
        d_W = ctx.array(w.T if what == "ABt" else w)
        if what == "AtB":
            D.upload(rng.standard_normal((M, N), dtype=np.float32) if value is None else np.full((M, N), value, np.float32))
        print("diverged", what, M, K, N, name, flush=True)
        for _ in range(4):
            ctx.sync()
            t = time.perf_counter()
            if what == "forward":
                ctx.nin_forward(A, d_W, B, None, out, M, K, N, 1.0, scn.NOSIGMOID, scn.FP32_PLANES)
            elif what == "ABt":  # [M x 256] times the transpose of [512 x 256]
                ctx.sgemm_ABt(A, d_W, out, M, K, N, ws)
            else:
                ctx.sgemm_AtB(A, D, dW, M, K, N)
            ctx.sync()
            best[name] = min(best.get(name, 1e9), 1e6 * (time.perf_counter() - t))
        got = (dW if what == "AtB" else out).download()
        assert np.isfinite(got).all() if value is None else not np.isfinite(got).any()
    print("us", {k: round(v) for k, v in best.items()}, flush=True)
    # (launches and waits are some 50 us of each)
    assert best["nan"] <= 5 * best["sound"] + 50 and best["inf"] <= 15 * best["sound"] + 50


@pytest.mark.parametrize("M,K,N", [(14000, 1728, 64), (30000, 256, 96), (20000, 512, 160)])
def test_planes_round_less_than_the_fp32_mfma(scn, ctx, M, K, N):
    """root mean square error against float64: 0.31 to 0.38 of the fp32 MFMA kernels' on these shapes, none of them
    a long contraction or few rows"""
    rng = np.random.default_rng(M)
    A, W = np.maximum(rng.standard_normal((M, K), dtype=np.float32), 0), rng.standard_normal((K, N), dtype=np.float32)
    want, err = A.astype(np.float64) @ W.astype(np.float64), []
    d_A, d_W, d_B, out = ctx.array(A), ctx.array(W), ctx.array(np.zeros(N, np.float32)), ctx.empty((M, N), np.float32)
    for p in (scn.FP32, scn.FP32_PLANES):
        ctx.nin_forward(d_A, d_W, d_B, None, out, M, K, N, 1.0, scn.NOSIGMOID, p)
        err.append(np.sqrt(((out.download() - want) ** 2).mean()))
    assert 0 < err[1] <= 0.5 * err[0]


# tiles, split contraction, weight gradient
@pytest.mark.parametrize("what,M", [("forward", 30000), ("forward", 200), ("AtB", 30000)])
@pytest.mark.parametrize("exponent", [-105, -112, -120, -130])
def test_operands_below_the_range_of_the_lower_planes(scn, ctx, what, M, exponent):
    """bf16 resolves 2^-133: of an operand so small that its lowest plane lies below that, 2^-134 is left out at most"""
    rng = np.random.default_rng(M - exponent)
    K, N = 256, 96
    tiny = (rng.standard_normal((M, K)) * 2.0 ** exponent).astype(np.float32)
    other = rng.standard_normal((K, N) if what == "forward" else (M, N)).astype(np.float32)
    if what == "forward":
        out = ctx.empty((M, N), np.float32)
        ctx.nin_forward(ctx.array(tiny), ctx.array(other), ctx.array(np.zeros(N, np.float32)), None, out, M, K, N, 1.0,
                        scn.NOSIGMOID, scn.FP32_PLANES)
        a, length = tiny, K
    else:
        out = ctx.array(np.zeros((K, N), np.float32))
        ctx.sgemm_AtB(ctx.array(tiny), ctx.array(other), out, M, K, N)
        a, length = tiny.T, M
    a, b = a.astype(np.float64), other.astype(np.float64)
    # what is left out of each operand, the rounding of the sums as for ordinary operands, and fp32's own grid
    allowed = 2.0 ** -134 * np.abs(b).sum(0) + 2e-6 * (np.abs(a) @ np.abs(b)) + length * 2.0 ** -149
    assert np.all(np.abs(out.download() - a @ b) <= allowed)


def test_a_context_without_room_for_weights_gives_the_same_bits(scn, ctx):
    import ctypes as C
    h = C.c_void_p()
    assert scn.lib().scn_ctx_create_for_plans(0, C.byref(h)) == scn.OK
    plain = scn.Context(handle=h.value)
    rng = np.random.default_rng(4)
    M, N = 60000, 256
    for K in (512, 1728):
        A, W = ctx.array(rng.standard_normal((M, K), dtype=np.float32)), ctx.array(rng.standard_normal((K, N), dtype=np.float32))
        D, B, ws = ctx.array(rng.standard_normal((M, N), dtype=np.float32)), ctx.array(np.zeros(N, np.float32)), ctx.empty(
            scn.lib().scn_sgemm_ABt_workspace(N, K), np.float32)
        outs = [(ctx.empty((M, N), np.float32), ctx.empty((M, N), np.float32), ctx.empty((M, K), np.float32)) for _ in range(2)]
        for c, (a, b, d) in zip((ctx, plain), outs):
            c.nin_forward(A, W, B, None, a, M, K, N, 1.0, scn.RELU, scn.FP32_PLANES)
            c.nin_forward(A, W, B, None, b, M, K, N, 1.0, scn.RELU, scn.BF16)
            c.sgemm_ABt(D, W, d, M, N, K, ws)
            c.sync()
        assert all(np.array_equal(x.download(), y.download()) for x, y in zip(*outs))
    scn.lib().scn_ctx_destroy(h)


@pytest.mark.parametrize("M,N,K", [(60000, 256, 512), (20001, 64, 100), (20001, 96, 36), (40001, 128, 260)])
def test_scratch_that_begins_at_any_float(scn, ctx, M, N, K):
    """a context without room for weights transposes W into the caller's scratch, wherever that begins"""
    import ctypes as C
    h = C.c_void_p()
    assert scn.lib().scn_ctx_create_for_plans(0, C.byref(h)) == scn.OK
    plain = scn.Context(handle=h.value)
    rng = np.random.default_rng(K)
    D, W = ctx.array(rng.standard_normal((M, N), dtype=np.float32)), ctx.array(rng.standard_normal((K, N), dtype=np.float32))
    room = ctx.empty(scn.lib().scn_sgemm_ABt_workspace(N, K) + 4, np.float32)
    got = []
    print("scratch", M, N, K, flush=True)
    for c, at in ((ctx, 0), (plain, 0), (plain, 1), (plain, 2)):
        out = ctx.empty((M, K), np.float32)
        ctx.sync()
        scn._check(scn.lib().scn_sgemm_ABt(c.h, D.ptr, W.ptr, out.ptr, M, N, K, C.c_void_p(room.ptr + 4 * at)))
        c.sync()
        got.append(out.download())
    f64 = D.download()[:500].astype(np.float64) @ W.download().astype(np.float64).T
    scale = np.abs(D.download()[:500]).astype(np.float64) @ np.abs(W.download()).astype(np.float64).T
    # (fp32's own accumulation, or the planes': a rounding every few of the N)
    assert all(np.all(np.abs(g[:500] - f64) <= 2e-6 * scale) for g in got)
    if N >= 256:  # the planes whatever the scratch
        assert all(np.array_equal(got[0], g) for g in got[1:])
    scn.lib().scn_ctx_destroy(h)
