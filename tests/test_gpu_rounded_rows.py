"""Rows that a pooling leaves rounded to bf16 beside its output: the contraction's bits are those of fp32 rows, which it
rounds itself, in every kernel that takes them."""
import ctypes as C

import numpy as np
import pytest

import brute
from test_gpu_capture import Graph
from test_gpu_run_ahead import _one_plan

pytestmark = pytest.mark.gpu


def rounded(v):  # to the nearest bf16, ties to the even one
    u = np.ascontiguousarray(v, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7fff + (u >> 16 & 1)) >> 16).astype(np.uint16)


@pytest.mark.parametrize("rows,out,ps,C", [(300, 1, 4, 8), (3000, 777, 9, 32), (500, 2000, 8, 160), (900, 63, 5, 12)])
def test_the_pooling_rounds(scn, ctx, rows, out, ps, C):
    rng = np.random.default_rng(C)
    d_in, rules = ctx.array(rng.standard_normal((rows, C), dtype=np.float32)), rng.integers(-1, rows, (out, ps)).astype(np.int32)
    d_rules = ctx.array(rules)
    a, b = [(ctx.array(np.full((out + 5, C), 7, np.float32)), ctx.array(np.full((out + 5, C), 7, np.int32))) for _ in range(2)]
    d16 = ctx.array(np.full((out + 5, C // 2), 7, np.int32))
    ctx.maxpool(d_in, a[0], d_rules, out, ps, C, a[1])
    ctx.maxpool_rounded(d_in, rows, b[0], d16, d_rules, out, ps, C, b[1])
    got = b[0].download()
    assert np.array_equal(a[0].download(), got) and np.array_equal(a[1].download(), b[1].download())
    half = d16.download()
    assert np.array_equal(half[:out].view(np.uint16).reshape(out, C), rounded(got[:out])) and np.all(half[out:] == 7)
    assert scn.lib().scn_maxpool_rounded(ctx.h, d_in.ptr, rows, b[0].ptr, d16.ptr, d_rules.ptr, out, ps, 6, b[1].ptr) != 0


# (rows, fs, nIn, N) few rows, by the split contractions, by lines, by rings of a wavefront's own; long ones of few rows
@pytest.mark.parametrize("rows,fs,nIn,N", [(40, 4, 64, 96), (900, 4, 320, 480), (26000, 4, 160, 320), (41600, 4, 64, 96), (10500, 4, 480, 640),
                                           (6001, 4, 384, 256), (20003, 27, 64, 128), (9000, 8, 32, 64)])
def test_the_bits_of_fp32_rows(scn, ctx, rows, fs, nIn, N):
    rng = np.random.default_rng(rows)
    K, n = fs * nIn, 1200
    x = rng.standard_normal((n, nIn), dtype=np.float32)
    d_x, d_x16 = ctx.array(x), ctx.array(rounded(x).view(np.int32))
    d_rules = ctx.array(rng.integers(-1, n, (rows, fs)).astype(np.int32))
    d_W = ctx.array((rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32))
    d_B, d_slopes = (ctx.array(rng.uniform(0.1, 0.4, N).astype(np.float32)) for _ in range(2))
    image, room = ctx.empty((-(-N // 32) * 32 * K * 2 // 4,), np.float32), ctx.empty((n, nIn // 2), np.float32)
    ctx.weight_images_many([(d_W, image, K, N, 0, scn.BF16)])
    outs = [ctx.array(np.full((rows + 300, N), 7, np.float32)) for _ in range(5)]
    print("rounded rows", rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward(d_x, d_rules, fs, nIn, d_W, d_B, d_slopes, outs[0], rows, N, 1.0, scn.PRELU, scn.BF16)
    ctx.conv_nin_forward_rounded(d_x, d_x16, d_rules, fs, nIn, d_W, image, d_B, d_slopes, outs[1], rows, N, 1.0, scn.PRELU)
    ctx.conv_nin_forward_rounded(d_x, d_x16, d_rules, fs, nIn, d_W, None, d_B, d_slopes, outs[2], rows, N, 1.0, scn.PRELU)
    ctx.conv_nin_forward_a16(d_x, n, room, d_rules, fs, nIn, d_W, d_B, d_slopes, outs[3], rows, N, 1.0, scn.PRELU)
    with Graph(ctx) as g:
        ctx.conv_nin_forward_rounded(d_x, d_x16, d_rules, fs, nIn, d_W, image, d_B, d_slopes, outs[4], rows, N, 1.0, scn.PRELU)
    for _ in range(2):
        g.replay(ctx)
    got = [o.download() for o in outs]
    g.close()
    assert all(np.array_equal(o, got[0]) and np.all(o[rows:] == 7) for o in got)


def test_a_net_of_bf16_operands(scn):
    """batches whose convolutions read rounded rows, and a small one whose do not: the bits of the pass that gathers"""
    from perf import cases
    runs = []
    for fused in (False, True):
        case = dict(name="wide", kind="net", stack="wide", batch=70, precision="bf16", fused=fused)
        s = cases.prepare(case, 3)
        out = [cases.run(s).copy() for _ in range(3)]
        assert all(np.array_equal(o, out[0]) for o in out)
        small = cases._prepare_net(dict(case, batch=2), 4)
        runs.append(np.concatenate([out[0], cases._run_net(small).copy()]))
    assert np.isfinite(runs[0]).all() and np.array_equal(runs[0], runs[1])


# (a contraction split over few rows, tiles, k_nin_rows16)
@pytest.mark.parametrize("nIn,N,densities", [(64, 96, (0.02, 0.02, 0.01)), (256, 320, (0.4, 0.4, 0.2, 0.42)),
                                             (512, 128, (0.5, 0.5, 0.35, 0.6))])
def test_rounded_rows_ahead_of_their_counts(scn, ctx, nIn, N, densities):
    """rows known on the device only: a pooling that rounds, and contractions of rounded rows, as with known counts"""
    rng = np.random.default_rng(nIn)
    fs, src, out = 4, scn.Grids(ctx), scn.Grids(ctx)
    d_W = ctx.array((rng.standard_normal((fs * nIn, N)) * np.sqrt(0.5 / nIn)).astype(np.float32))
    d_B = ctx.array(rng.uniform(-0.5, 0.5, N).astype(np.float32))
    rounds = []
    for i, density in enumerate(densities):
        samples, nSites = brute.random_samples(rng, 30, 2, 41, density)
        x = rng.standard_normal((nSites, nIn), dtype=np.float32)
        d_x, d_x16, room = ctx.array(x), ctx.array(rounded(x).view(np.int32)), ctx.empty((nSites, nIn // 2), np.float32)
        rules, bound = _one_plan(scn, ctx, src, out, samples, nSites, i > 0)
        outs = [ctx.array(np.full((bound, N), 7, np.float32)) for _ in range(2)]
        pooled = [ctx.array(np.full((bound, c), 7, t)) for c, t in ((nIn, np.float32), (nIn // 2, np.int32), (nIn, np.int32))]
        print("rounded rows ahead", nIn, N, density, bound, flush=True)
        assert scn.lib().scn_ctx_rows_from(ctx.h, out.h) == scn.OK
        ctx.maxpool_rounded(d_x, nSites, *pooled[:2], rules, bound, fs, nIn, pooled[2])
        ctx.conv_nin_forward_rounded(d_x, d_x16, rules, fs, nIn, d_W, None, d_B, None, outs[0], bound, N)
        ctx.conv_nin_forward_a16(d_x, nSites, room, rules, fs, nIn, d_W, d_B, None, outs[1], bound, N)
        scn.lib().scn_ctx_rows_from(ctx.h, None)
        assert scn.settle(ctx)
        held = C.c_int()
        assert scn.lib().scn_ctx_rows_held(ctx.h, C.byref(held)) == scn.OK
        n = out.info()["nSpatialSites"]
        known = [ctx.array(np.full((n, c), 7, t)) for c, t in ((nIn, np.float32), (nIn // 2, np.int32), (nIn, np.int32), (N, np.float32))]
        ctx.maxpool_rounded(d_x, nSites, *known[:2], rules, n, fs, nIn, known[2])
        ctx.conv_nin_forward(d_x, rules, fs, nIn, d_W, d_B, None, known[3], n, N, 1.0, scn.RELU, scn.BF16)
        for a, b in zip(pooled, known):
            a = a.download()
            assert np.array_equal(a[:n], b.download()) and np.all(a[n:] == 7)
        want = known[3].download()
        for a in outs:
            a = a.download()
            assert np.all(a[n:] == 7)
            if held.value:
                assert np.array_equal(a[:n], want), (i, n, bound)
            else:  # two orders of summation of the same K products
                scale = np.abs(x).max() * np.abs(d_W.download()).sum(0).max() + 0.5
                assert np.abs(a[:n] - want).max() <= 2 * fs * nIn * 2.0 ** -24 * scale
        rounds.append(held.value)
    assert rounds[:2] == [1, 1]


def test_an_epoch_of_bf16_operands(scn):
    """The poolings of a training batch round, too: an epoch of one batch, whose convolutions are left out and read rounded
    rows, costs what the batch by itself, which gathers, costs, and leaves its gradients."""
    from sparseconvnet_archived_amd import hostapi, synthetic
    batch = 70
    cfg = synthetic.config(4, batch=batch)
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TRAINBATCH)
    for pts, f, label in synthetic.make_samples(cfg, 44):
        ds.add_points(cfg.dimension, cfg.lattice, pts, f, label)
    costs, left, pay = [], [], 0
    for epoch in (True, False):
        net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, threads=1)
        cfg.build(net)
        net.setPrecision(scn.BF16)
        for i, (W, B, pr) in synthetic.he_normal_weights(net.layers(), 45).items():
            net.set_weights(i, W, B, pr)
        net.set_training(0.01, 0.9, shuffle=False)
        if epoch:
            costs.append(net.processDatasetTrain(ds, batch, 0.01, 0.9))
        else:
            net.begin(ds, batch)
            assert net.next_batch()
            costs.append(net.batch_outputs()["nll"] / batch)
            for i, l in enumerate(net.layers()):
                if l["kind"].startswith("nin") and i > 1 and l["nIn"] % 4 == 0:
                    rows = net.interface(i + 1, want_features=False)["nSpatialSites"]
                    pay += scn.lib().scn_rounded_rows_pay(C.c_void_p(net.context_handle()), rows, 4, l["nIn"] // 4, l["nOut"])
            net.end()
        left.append([net.get_weights(i, True) for i, l in enumerate(net.layers()) if l["kind"].startswith("nin")])
        net.close()
    assert pay >= 2  # (layers whose rows come rounded)
    print("costs", costs, "gradients", [[float(np.linalg.norm(u - v) / np.linalg.norm(v)) for u, v in zip(a, b) if v is not None]
                                        for a, b in zip(*left)], flush=True)
    assert abs(costs[0] - costs[1]) <= 1e-6 * abs(costs[1])
    # (the same bits forward; sums of up to 10^5 products in another order backward, through six layers: sqrt(1e5) 2^-24 each)
    for a, b in zip(*left):
        for u, v in zip(a, b):
            assert v is None or np.linalg.norm(u - v) <= 6 * 2e-5 * np.linalg.norm(v)
