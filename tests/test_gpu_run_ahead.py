"""A resident batch's layers queued behind its rule books, their numbers of rows read on the device: whatever batches
came before, the probabilities and the multiply-adds are those of a net that has seen no other batch (which waits for
its counts), bit for bit."""
import ctypes as C

import numpy as np
import pytest

import brute
from gpu_util import flatten_samples

pytestmark = pytest.mark.gpu


def _net(cfg, weights, fused):
    from sparseconvnet_archived_amd import hostapi
    net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, nTop=1, threads=1)
    cfg.build(net)
    net.setFusedConvolutions(fused)
    for i, (W, B, pr) in (weights or {}).items():
        net.set_weights(i, W, B, pr)
    return net


# (samples of the batches in turn: the bounds hold, are outgrown, and are far too wide; kernels of few rows and of many)
@pytest.mark.parametrize("config,sizes,fused,bf16", [(2, (3, 3, 40, 1, 40, 2), True, False), (2, (30, 30, 5), False, False),
                                                     (2, (8, 9, 60, 7), True, True), (3, (2, 2, 9, 1), True, False)])
def test_layers_ahead_of_the_counts(scn, config, sizes, fused, bf16):
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(config, batch=max(sizes))
    net = _net(cfg, None, fused)
    weights = synthetic.he_normal_weights(net.layers(), 5)
    net.close()
    net = _net(cfg, weights, fused)
    ctx = scn.Context(handle=net.context_handle())
    for i, b in enumerate(sizes):
        S, K, R, bg, feats, n = synthetic.codify(synthetic.make_samples(cfg, 300 + i, batch=b), cfg.dimension, cfg.lattice,
                                                 net.inputSpatialSize, cfg.nInputFeatures)
        got = []
        for use in (net, _net(cfg, weights, fused)):
            use.setPrecision(scn.BF16 if bf16 else scn.FP32)
            d = [ctx.array(S, np.int32), ctx.array(K, np.int64), ctx.array(R, np.int32), ctx.array(bg, np.int32),
                 ctx.array(feats, np.float32)]
            ctx.sync()
            p = np.zeros((b, cfg.nClasses), np.float32)
            hostapi.take_multiply_add_count()
            use.forward_resident(b, d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, len(K), n, d[4].ptr, p)
            got.append((p, hostapi.take_multiply_add_count(), use.interface(2), use.interface(6)))
            if use is not net:
                use.close()
        a, w = got
        assert np.isfinite(a[0]).all() and np.array_equal(a[0], w[0]), (i, b)
        assert a[1] == w[1] > 0, (i, b)
        for x, y in zip(a[2:], w[2:]):
            assert x["nSpatialSites"] == y["nSpatialSites"] and np.array_equal(x["features"], y["features"]), (i, b)
    net.close()


def _one_plan(scn, ctx, src, out, samples, nSites, record):
    """the rule book of a side-2 window over a 41^2 field, deferred or not -> (rules, rows or their bound)"""
    scn.clear_many(ctx, [src, out])
    src.build(len(samples), 2, 41, *flatten_samples(samples), nSites)
    if record:
        scn.defer_counts(ctx, True)
        scn.chain_rules(ctx, True)
    _, rules, n, w = scn.rules_square(ctx, src, 41, 40, 2, 1, 1, out=out)
    if record:
        scn.chain_rules(ctx, False)
        scn.defer_counts(ctx, False)
    return rules, n


def test_fp32_waits_for_its_rows_and_chooses_by_them(scn, ctx):
    """SCN_FP32 takes the planes for few rows and for long contractions: queued behind a plan whose bound says otherwise,
    it gives the bits of the rows that there are."""
    rng = np.random.default_rng(12)
    # (few rows under a wide bound; a bound of some 11000 rows makes a long contraction, 3900 of them do not)
    for nIn, N, densities in ((32, 320, (0.08, 0.08, 0.02)), (1024, 1024, (0.5, 0.5, 0.12))):
        fs, src, out = 4, scn.Grids(ctx), scn.Grids(ctx)
        d_W = ctx.array((rng.standard_normal((fs * nIn, N)) * 0.1).astype(np.float32))
        d_B = ctx.array(rng.uniform(-0.5, 0.5, N).astype(np.float32))
        for i, density in enumerate(densities):
            samples, nSites = brute.random_samples(rng, 6, 2, 41, density)
            d_in = ctx.array(rng.standard_normal((nSites, nIn)).astype(np.float32))
            rules, bound = _one_plan(scn, ctx, src, out, samples, nSites, i > 0)
            got = ctx.array(np.full((bound, N), 7, np.float32))
            print("fp32 ahead", density, nIn, bound, flush=True)
            assert scn.lib().scn_ctx_rows_from(ctx.h, out.h) == scn.OK
            ctx.conv_nin_forward(d_in, rules, fs, nIn, d_W, d_B, None, got, bound, N, 1.0, scn.RELU, scn.FP32)
            scn.lib().scn_ctx_rows_from(ctx.h, None)
            assert scn.settle(ctx)
            held = C.c_int()
            assert scn.lib().scn_ctx_rows_held(ctx.h, C.byref(held)) == scn.OK and held.value == 1
            n = out.info()["nSpatialSites"]
            known = ctx.array(np.full((n, N), 7, np.float32))
            ctx.conv_nin_forward(d_in, rules, fs, nIn, d_W, d_B, None, known, n, N, 1.0, scn.RELU, scn.FP32)
            assert np.array_equal(got.download()[:n], known.download()), (density, n, bound)


def test_settled_counts_are_no_longer_read_on_the_device(scn, ctx):
    """scn_ctx_rows_from ends with the settling (and with its grids): a call of more rows takes its own number."""
    rng = np.random.default_rng(13)
    nIn, N, fs, M = 32, 320, 4, 5000
    src, out = scn.Grids(ctx), scn.Grids(ctx)
    A, W, B = (ctx.array(rng.standard_normal(s, dtype=np.float32)) for s in ((M, fs * nIn), (fs * nIn, N), (N,)))
    known = ctx.empty((M, N), np.float32)
    ctx.nin_forward(A, W, B, None, known, M, fs * nIn, N, 1.0, scn.RELU, scn.FP32_PLANES)
    for end in ("settle", "destroy"):
        for i in range(2):
            samples, nSites = brute.random_samples(rng, 6, 2, 41, 0.02)
            _one_plan(scn, ctx, src, out, samples, nSites, i > 0)
        assert scn.lib().scn_ctx_rows_from(ctx.h, out.h) == scn.OK
        if end == "settle":
            assert scn.settle(ctx)
        else:
            out.close()
        got = ctx.array(np.full((M, N), 7, np.float32))
        ctx.nin_forward(A, W, B, None, got, M, fs * nIn, N, 1.0, scn.RELU, scn.FP32_PLANES)
        assert np.array_equal(got.download(), known.download()), end
    assert scn.lib().scn_rules_settle(ctx.h) == scn.OK


@pytest.mark.parametrize("M", [200, 20000])  # split contraction, tiles
def test_backward_products_keep_their_own_rows(scn, ctx, M):
    """scn_ctx_rows_from speaks to the forward calls: a product with W^T meanwhile computes the rows it is given."""
    rng = np.random.default_rng(14)
    N, K = 256, 128
    src, out = scn.Grids(ctx), scn.Grids(ctx)
    D, W = ctx.array(rng.standard_normal((M, N), dtype=np.float32)), ctx.array(rng.standard_normal((K, N), dtype=np.float32))
    ws, outs = ctx.empty(N * K + K, np.float32), [ctx.array(np.full((M, K), 7, np.float32)) for _ in range(2)]
    ctx.sgemm_ABt(D, W, outs[0], M, N, K, ws)
    for i in range(2):
        _one_plan(scn, ctx, src, out, *brute.random_samples(rng, 2, 2, 41, 0.003), i > 0)
    assert scn.lib().scn_ctx_rows_from(ctx.h, out.h) == scn.OK
    ctx.sgemm_ABt(D, W, outs[1], M, N, K, ws)
    scn.lib().scn_ctx_rows_from(ctx.h, None)
    assert scn.settle(ctx) and out.info()["nSpatialSites"] < M
    assert np.array_equal(outs[0].download(), outs[1].download())


# split contraction up to 1248 rows (three planes) and 1792 (one), tiles above: dense batches lie above, sparse ones below
@pytest.mark.parametrize("precision", ["FP32_PLANES", "BF16"])
def test_a_wrong_guess_of_rows_leaves_none_out(scn, ctx, precision):
    """Batches on both sides of the line between two kernels, each queued by the rows of the one before: every row is
    computed, and where scn_ctx_rows_held says so it is the row that known counts give, bit for bit."""
    p = getattr(scn, precision)
    rng = np.random.default_rng(11)
    nIn, N, fs = 32, 320, 4
    src, out = scn.Grids(ctx), scn.Grids(ctx)
    W = (rng.standard_normal((fs * nIn, N)) * 0.1).astype(np.float32)
    d_W, d_B = ctx.array(W), ctx.array(rng.uniform(-0.5, 0.5, N).astype(np.float32))
    seen = []
    for i, density in enumerate((0.08, 0.08, 0.02, 0.02, 0.08, 0.08, 0.02)):
        samples, nSites = brute.random_samples(rng, 6, 2, 41, density)
        inp = rng.standard_normal((nSites, nIn)).astype(np.float32)
        d_in = ctx.array(inp)
        rules, bound = _one_plan(scn, ctx, src, out, samples, nSites, i > 0)
        got = ctx.array(np.full((bound, N), 7, np.float32))
        print("rows ahead", precision, density, bound, flush=True)
        assert scn.lib().scn_ctx_rows_from(ctx.h, out.h) == scn.OK
        ctx.conv_nin_forward(d_in, rules, fs, nIn, d_W, d_B, None, got, bound, N, 1.0, scn.RELU, p)
        scn.lib().scn_ctx_rows_from(ctx.h, None)
        assert scn.settle(ctx)
        held = C.c_int()
        assert scn.lib().scn_ctx_rows_held(ctx.h, C.byref(held)) == scn.OK
        n = out.info()["nSpatialSites"]
        known = ctx.array(np.full((n, N), 7, np.float32))
        ctx.conv_nin_forward(d_in, rules, fs, nIn, d_W, d_B, None, known, n, N, 1.0, scn.RELU, p)
        a, b = got.download(), known.download()
        # two orders of summation of the same products: a rounding of each of the K partial sums at most
        assert np.abs(a[:n] - b).max() <= 2 * fs * nIn * 2.0 ** -24 * (np.abs(inp).max() * np.abs(W).sum(0).max() + 0.5)
        assert (a[n:] == 7).all()
        assert not held.value or np.array_equal(a[:n], b), (i, n)
        seen.append(held.value)
    # wrong where the density changed and right where it did not
    assert seen == [1, 1, 0, 1, 0, 1, 0]
    # a settling that settles nothing speaks of no earlier pass
    assert scn.settle(ctx) and scn.lib().scn_ctx_rows_held(ctx.h, C.byref(held)) == scn.OK and held.value == 1


def test_the_second_batch_finds_room_in_the_firsts_buffers(scn):
    """The bounds that a pass ahead of its counts is queued with fit the buffers that the first batch has left: none is
    allocated anew for a batch of the same kind (each a wait for the device)."""
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(2, batch=100)
    net = _net(cfg, None, False)
    weights = synthetic.he_normal_weights(net.layers(), 5)
    net.close()
    net = _net(cfg, weights, False)
    ctx = scn.Context(handle=net.context_handle())
    hip, free = C.CDLL("libamdhip64.so"), []
    batches = []
    for i in range(3):
        S, K, R, bg, feats, n = synthetic.codify(synthetic.make_samples(cfg, 400 + i), cfg.dimension, cfg.lattice,
                                                 net.inputSpatialSize, cfg.nInputFeatures)
        batches.append(([ctx.array(S, np.int32), ctx.array(K, np.int64), ctx.array(R, np.int32), ctx.array(bg, np.int32)],
                        len(K), n, ctx.array(feats, np.float32)))
    for d, k, n, f in batches:
        p = np.zeros((100, cfg.nClasses), np.float32)
        net.forward_resident(100, d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, k, n, f.ptr, p)
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        free.append(a.value)
    net.close()
    print("free memory taken", free[0] - free[1], free[1] - free[2], flush=True)
    # (the layers' buffers anew were 48 MB; the second batch's recorded plans need some masks and tables of their own)
    assert free[0] - free[1] <= 8 << 20 and free[1] == free[2]


def test_wrong_guesses_over_a_net(scn):
    """Drawings of few strokes and of many in turn: the guess of the first layer's rows lies on the other side of the line
    between its kernels time and again, the pass is queued once more, and the bits stay those of a net that has seen no
    other drawing."""
    from sparseconvnet_archived_amd import synthetic
    cfg = synthetic.config(2, batch=1)
    net = _net(cfg, None, True)
    weights = synthetic.he_normal_weights(net.layers(), 5)
    net.close()
    net = _net(cfg, weights, True)
    ctx = scn.Context(handle=net.context_handle())
    rng = np.random.default_rng(21)
    held = []
    for i, target in enumerate((460, 440, 110, 450, 120, 100, 460, 430)):
        pts = np.asarray(synthetic.strokes(rng, cfg.lattice, target), np.int32)
        sample = [(pts, rng.uniform(-1, 1, (len(pts), 3)).astype(np.float32), 0)]
        S, K, R, bg, feats, n = synthetic.codify(sample, cfg.dimension, cfg.lattice, net.inputSpatialSize, cfg.nInputFeatures)
        d = [ctx.array(S, np.int32), ctx.array(K, np.int64), ctx.array(R, np.int32), ctx.array(bg, np.int32),
             ctx.array(feats, np.float32)]
        fresh, got = _net(cfg, weights, True), []
        for use in (net, fresh):
            p = np.zeros((1, cfg.nClasses), np.float32)
            use.forward_resident(1, d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, len(K), n, d[4].ptr, p)
            got.append((p, use.interface(2)["features"], use.interface(6)["features"]))
            if use is net:
                h = C.c_int()
                assert scn.lib().scn_ctx_rows_held(ctx.h, C.byref(h)) == scn.OK
                held.append(h.value)
        fresh.close()
        assert all(np.array_equal(a, b) for a, b in zip(*got)), (i, target)
    net.close()
    # (the first drawing's counts are known, the next is guessed by it)
    assert held[:2] == [1, 1] and held.count(0) >= 3 and held.count(1) >= 4, held


def test_a_bound_beyond_32_bit_choices_is_no_batch_beyond_them(scn):
    """A layer in front of a pooling with 1.8 of the 2.1 billion elements that 32-bit choices index: a quarter more, its
    bound in the next batch, passes them.  That batch waits for its counts and is taken as the first one was."""
    from sparseconvnet_archived_amd import hostapi, synthetic
    rng = np.random.default_rng(6)
    batch, field = 200, 41
    net = hostapi.Net(2, 1, 2, threads=1)
    net.addLeNetLayerMP(8192, 2, 1, 2, 2, scn.RELU)
    net.addTerminalPoolingLayer(20)
    net.addSoftmaxLayer()
    net.setFusedConvolutions(True)
    assert net.inputSpatialSize == field
    for i, (W, B, pr) in synthetic.he_normal_weights(net.layers(), 5).items():
        net.set_weights(i, W, B, pr)
    ctx = scn.Context(handle=net.context_handle())
    samples, n = brute.random_samples(rng, batch, 2, field, 0.26)
    S, K, R, bg = flatten_samples(samples)
    feats = rng.standard_normal((n, 1)).astype(np.float32)
    d = [ctx.array(S, np.int32), ctx.array(K, np.int64), ctx.array(R, np.int32), ctx.array(bg, np.int32), ctx.array(feats)]
    got = []
    for _ in range(3):
        p = np.zeros((batch, 2), np.float32)
        print("a batch of 1.8e9 elements", flush=True)
        net.forward_resident(batch, d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, len(K), n, d[4].ptr, p)
        got.append(p)
    rows = net.interface(2, want_features=False)["nSpatialSites"]
    net.close()
    assert 1.75e9 < rows * 8192 < 2 ** 31 < 1.25 * rows * 8192
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


def test_a_first_layer_and_its_matrix_ahead_of_their_rows(scn, ctx):
    """scn_conv_nin_forward_matrix with rows known on the device: matrix and layer of the rows that there are, whichever way
    the guess of them sent it (few rows: two launches; more: one)"""
    rng = np.random.default_rng(15)
    for nIn, N, fs, densities in ((3, 32, 4, (0.3, 0.3, 0.1, 0.02)), (3, 32, 4, (0.004, 0.004, 0.003))):
        src, out = scn.Grids(ctx), scn.Grids(ctx)
        d_W, d_B = (ctx.array(rng.standard_normal(s, dtype=np.float32)) for s in ((fs * nIn, N), (N,)))
        for i, density in enumerate(densities):
            samples, nSites = brute.random_samples(rng, 6, 2, 41, density)
            inp = rng.standard_normal((nSites, nIn)).astype(np.float32)
            d_in = ctx.array(inp)
            rules, bound = _one_plan(scn, ctx, src, out, samples, nSites, i > 0)
            matrix, got = ctx.array(np.full((bound, fs * nIn), 7, np.float32)), ctx.array(np.full((bound, N), 7, np.float32))
            print("matrix ahead", density, bound, flush=True)
            assert scn.lib().scn_ctx_rows_from(ctx.h, out.h) == scn.OK
            scn._check(scn.lib().scn_conv_nin_forward_matrix(ctx.h, d_in.ptr, rules.ptr, fs, nIn, matrix.ptr, d_W.ptr, d_B.ptr, None,
                                                             got.ptr, bound, N, 1.0, scn.RELU, scn.FP32_PLANES))
            scn.lib().scn_ctx_rows_from(ctx.h, None)
            assert scn.settle(ctx)
            held = C.c_int()
            assert scn.lib().scn_ctx_rows_held(ctx.h, C.byref(held)) == scn.OK
            n = out.info()["nSpatialSites"]
            r = rules.download().reshape(-1, fs)[:n]
            dense = np.where(r[:, :, None] >= 0, inp[np.maximum(r, 0)], 0).reshape(n, fs * nIn)
            assert np.array_equal(matrix.download()[:n], dense)
            known = ctx.array(np.full((n, N), 7, np.float32))
            ctx.nin_forward(ctx.array(dense), d_W, d_B, None, known, n, fs * nIn, N, 1.0, scn.RELU, scn.FP32_PLANES)
            if held.value:
                assert np.array_equal(got.download()[:n], known.download()), (density, n, bound)
            else:
                assert np.allclose(got.download()[:n], known.download(), rtol=1e-5, atol=1e-5)


def test_several_tiles_to_a_workgroup_ahead_of_their_rows(scn, ctx):
    """plain rows known on the device, more and fewer than the batch before had (k_nin_lines' LONG)"""
    rng = np.random.default_rng(16)
    K, N = 128, 128
    src, out = scn.Grids(ctx), scn.Grids(ctx)
    d_W, d_B = (ctx.array(rng.standard_normal(s, dtype=np.float32)) for s in ((K, N), (N,)))
    for i, density in enumerate((0.5, 0.5, 0.3, 0.6)):
        samples, nSites = brute.random_samples(rng, 30, 2, 41, density)
        _, bound = _one_plan(scn, ctx, src, out, samples, nSites, i > 0)
        A = ctx.array(rng.standard_normal((bound, K), dtype=np.float32))
        got = ctx.array(np.full((bound, N), 7, np.float32))
        print("several tiles ahead", density, bound, flush=True)
        assert scn.lib().scn_ctx_rows_from(ctx.h, out.h) == scn.OK
        ctx.nin_forward(A, d_W, d_B, None, got, bound, K, N, 1.0, scn.RELU, scn.FP32_PLANES)
        scn.lib().scn_ctx_rows_from(ctx.h, None)
        assert scn.settle(ctx)
        n = out.info()["nSpatialSites"]
        known = ctx.array(np.full((n, N), 7, np.float32))
        ctx.nin_forward(A, d_W, d_B, None, known, n, K, N, 1.0, scn.RELU, scn.FP32_PLANES)
        assert np.array_equal(got.download()[:n], known.download()), (density, n, bound)
        assert np.all(got.download()[n:] == 7)
