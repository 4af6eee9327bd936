"""The gradient of a pooling's input by rows, through its rules turned round, and with it the sums over the background of
the convolution before: against the scatter that the choices stand for, in float64."""
import numpy as np
import pytest

from test_gpu_conv_backward import layer

pytestmark = pytest.mark.gpu


# one, two, four and eight windows to a row; a sample without sites and a full one (whose pooling's output is full, too);
# a channel group of 16 that is not whole, rows that are no whole workgroups; more windows a sample than are asked for at
# once (2-D, 90: a full sample has 1936); sums over 1, 4 and 8 positions, and none
@pytest.mark.parametrize("d,field,window,size,stride,batch,density,C,act", [
    (2, 10, 2, 3, 2, 4, 0.2, 32, "RELU"), (2, 9, 2, 2, 2, 5, 0.1, 4, "NOSIGMOID"), (3, 9, 2, 2, 2, 4, 0.05, 36, "RELU"),
    (3, 8, 2, 3, 2, 3, 0.1, 20, "LEAKYRELU"), (2, 8, 2, 2, 1, 3, 0.3, 64, None), (1, 20, 2, 3, 2, 6, 0.2, 12, "TANH"),
    (2, 90, 2, 3, 2, 3, 0.1, 32, "RELU"), (2, 9, 1, 3, 3, 4, 0.3, 300, "RELU"), (2, 14, 3, 2, 2, 40, 0.02, 32, "RELU")])
def test_pool_gradient(scn, ctx, d, field, window, size, stride, batch, density, C, act):
    rng = np.random.default_rng(field * size + C)
    g, n, _, fs, _, bg = layer(scn, ctx, d, field, window, batch, density, field + C)
    h, p = scn.Grids(ctx), scn.Grids(ctx)
    mid = field - window + 1
    inRows = g.plan_square(h, field, mid, window, 1)
    d_conv = ctx.empty((inRows, fs), np.int32)
    g.fill(h, d_conv, inRows * fs)
    out = (mid - size) // stride + 1
    width = size ** d
    rows = h.plan_square(p, mid, out, size, stride)
    d_rules = ctx.empty((rows, width), np.int32)
    h.fill(p, d_rules, rows * width)
    slots = scn.lib().scn_pool_inverse_slots(d, size, stride)
    assert slots == (-(-size // stride)) ** d
    print("pool gradient", d, field, window, size, stride, batch, C, "rows", rows, "of", inRows, flush=True)
    x = rng.standard_normal((inRows, C), dtype=np.float32)
    y, choice = ctx.empty((rows, C), np.float32), ctx.empty((rows, C), np.int32)
    ctx.maxpool(ctx.array(x), y, d_rules, rows, width, C, choice)
    D = rng.standard_normal((rows, C), dtype=np.float32)
    inverse, samples = ctx.array(np.full((inRows, slots), 7, np.int32)), ctx.array(np.full(2 * batch + 1, 7, np.int32))
    ctx.pool_inverse_many([(h, p, d_rules, inverse, samples, rows, inRows, size, stride)])
    rules = d_rules.download().astype(np.int64)
    got = samples.download()
    inBg = got[batch + 1:]
    assert got[0] == 0 and got[batch] == rows and np.all(np.diff(got[:batch + 1]) >= 0)
    isBg = np.zeros(inRows, bool)
    isBg[inBg[inBg >= 0]] = True
    inv = inverse.download()
    assert np.all(inv[isBg] == -2)
    for r in rng.choice(np.nonzero(~isBg)[0], min(200, int((~isBg).sum())), replace=False):
        assert sorted(w for w in inv[r] if w >= 0) == sorted(np.nonzero((rules == r).any(1))[0])
    for s in range(batch):  # the windows that name a sample's background lie in its range
        named = np.nonzero((rules == inBg[s]).any(1))[0] if inBg[s] >= 0 else []
        assert all(got[s] <= w < got[s + 1] for w in named)
    # the gradient, with and without sums
    ch, v = choice.download().astype(np.int64), D.astype(np.float64)
    o = y.download().astype(np.float64)
    if act == "RELU":
        v = v * (o > 0)
    elif act == "LEAKYRELU":
        v = np.where(o > 0, v, v * 0.01)
    elif act == "TANH":
        v = v * (1 + o) * (1 - o)
    want, size_of = np.zeros(inRows * C), np.zeros(inRows * C)
    np.add.at(want, ch[ch >= 0], v[ch >= 0])
    np.add.at(size_of, ch[ch >= 0], np.abs(v[ch >= 0]))
    want, size_of = want.reshape(inRows, C), size_of.reshape(inRows, C)
    background = ctx.empty(inRows + 2 * batch, np.int32)
    convInverse = ctx.empty((n, fs), np.int32)
    ctx.rules_inverse_many([(g, d_conv, convInverse, background, None, inRows, n, fs)])
    mask = background.download()[:inRows]
    first = np.searchsorted(np.arange(rows), got[:batch + 1])
    sums, sums_of = np.zeros((batch * fs, C)), np.zeros((batch * fs, C))
    for s in range(batch):
        w = slice(first[s], first[s + 1])
        row, col = np.where(ch[w] >= 0, ch[w] // C, 0), np.broadcast_to(np.arange(C), ch[w].shape)
        for f in range(fs):
            hit = (ch[w] >= 0) & ((mask[row] >> f) & 1 == 1)
            np.add.at(sums[s * fs + f], col[hit], v[w][hit])
            np.add.at(sums_of[s * fs + f], col[hit], np.abs(v[w][hit]))
    for withSums in (False, True) if fs <= 8 else (False,):
        din = ctx.array(np.full((inRows + batch * fs, C), 7, np.float32))
        ctx.maxpool_gradient(din, inRows, ctx.array(D), rows, C, choice, y if act else None,
                             getattr(scn, act) if act else scn.NOSIGMOID, inverse, slots, samples, batch,
                             background if withSums else None, fs if withSums else 0)
        res = din.download()
        # (the sums' longest chain: a lane's windows, six shuffles, eight wavefronts)
        assert np.all(np.abs(res[:inRows] - want) <= 4e-6 * size_of + 1e-30)
        assert np.all(res[inRows:] == 7) if not withSums else np.all(np.abs(res[inRows:] - sums) <= 4e-6 * sums_of + 1e-30)


def test_pool_gradient_refusals(scn, ctx):
    f = scn.lib().scn_pool_inverse_slots
    assert [f(2, 3, 1), f(3, 3, 1), f(2, 4, 2), f(3, 4, 2), f(0, 2, 2), f(2, 2, 0)] == [0, 0, 4, 8, 0, 0]
    b, i = ctx.empty((64, 64), np.float32), ctx.empty((64, 64), np.int32)
    for kw in (dict(C_=6), dict(slots=3), dict(act=scn.PRELU), dict(fs=9, d_background=i)):
        a = dict(d_din=b, inputRows=4, d_dout=b, rows=4, C_=4, d_choice=i, d_out=None, act=scn.NOSIGMOID, d_inverse=i, slots=1,
                 d_samples=i, batch=1)
        a.update(kw)
        with pytest.raises(scn.ScnError):
            ctx.maxpool_gradient(**a)


# drawings alike: all five poolings by rows.  One that fills its field among seven of few points, whose 2400 windows of the first
# pooling a workgroup would walk (the average is some 300): that one is scattered
@pytest.mark.parametrize("sides,turned", [([26] * 8, 5), ([5, 5, 5, 96, 5, 5, 5, 5], 4)])
def test_the_longest_sample_decides(scn, sides, turned):
    from sparseconvnet_archived_amd import hostapi, synthetic
    from test_gpu_training import pair, rel_l2
    cfg = synthetic.config(2, batch=8)
    rng = np.random.default_rng(sum(sides))
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TRAINBATCH)
    for side in sides:
        at = np.stack(np.meshgrid(np.arange(side), np.arange(side), indexing="ij"), -1).reshape(-1, 2) + (96 - side) // 2
        ds.add_points(2, cfg.lattice, at.astype(np.int32), rng.uniform(-1, 1, (side * side, 3)).astype(np.float32),
                      int(rng.integers(0, 100)))
    left = []
    for epoch in (True, False):  # (a batch by itself scatters everything)
        net, _ = pair(cfg, hostapi, 53)
        net.set_training(0.01, 0.9, shuffle=False)
        if epoch:
            net.processDatasetTrain(ds, 8, 0.01, 0.9)
        else:
            net.begin(ds, 8)
            assert net.next_batch()
        assert net.turned_poolings() == (turned if epoch else 0)
        left.append([a for i, l in enumerate(net.layers()) if l["kind"].startswith("nin")
                     for a in net.get_weights(i, momentum=True) if a is not None])
        net.close()
    for a, b in zip(*left):  # (the same forward pass, bit for bit: fp32 sums in other orders)
        assert rel_l2(a, b) <= 1e-5


def test_where_the_samples_begin_is_copied(scn, ctx):
    """two poolings' one behind the other; to pinned host memory as epochs have it, and nothing behind them"""
    items, keep, n = [], [], 7
    for field, size, stride in ((10, 3, 2), (13, 2, 2)):
        g, _, _, _, _, _ = layer(scn, ctx, 2, field, 2, n, 0.2, field)
        h, p = scn.Grids(ctx), scn.Grids(ctx)
        inRows = g.plan_square(h, field, field - 1, 2, 1)
        rows = h.plan_square(p, field - 1, (field - 1 - size) // stride + 1, size, stride)
        rules = ctx.empty((rows, size * size), np.int32)
        h.fill(p, rules, rows * size * size)
        slots = scn.lib().scn_pool_inverse_slots(2, size, stride)
        keep.append((g, h, p))
        items.append((h, p, rules, ctx.empty((inRows, slots), np.int32), ctx.empty(2 * n + 1, np.int32), rows, inRows, size, stride))
    copy = ctx.host_alloc(4 * 32)
    to = copy.buffer()
    host = np.frombuffer(to, np.int32)
    host[:] = 7
    ctx.pool_inverse_many(items, copy)
    ctx.sync()
    want = np.concatenate([i[4].download()[:n + 1] for i in items])
    assert np.array_equal(host[:2 * (n + 1)], want) and np.all(host[2 * (n + 1):32] == 7)


@pytest.mark.parametrize("d,field,size,stride,C", [(2, 30, 3, 2, 32), (3, 9, 2, 2, 20)])
@pytest.mark.parametrize("act", ["RELU", "LEAKYRELU", "TANH", None])
def test_pool_gradient_of_what_is_not_finite(scn, ctx, d, field, size, stride, C, act):
    """infinities, NaN and the type's largest in the gradient and in what is pooled: each goes to the row that was chosen and
    to the sums of its positions, and to nothing else"""
    rng = np.random.default_rng(field + C)
    batch = 4
    g, n, _, fs, _, _ = layer(scn, ctx, d, field, 2, batch, 0.15, 3)
    h, p = scn.Grids(ctx), scn.Grids(ctx)
    mid = field - 1
    inRows = g.plan_square(h, field, mid, 2, 1)
    d_conv = ctx.empty((inRows, fs), np.int32)
    g.fill(h, d_conv, inRows * fs)
    rows, width = h.plan_square(p, mid, (mid - size) // stride + 1, size, stride), size ** d
    d_rules = ctx.empty((rows, width), np.int32)
    h.fill(p, d_rules, rows * width)
    slots = scn.lib().scn_pool_inverse_slots(d, size, stride)
    x, D = rng.standard_normal((inRows, C), dtype=np.float32), rng.standard_normal((rows, C), dtype=np.float32)
    odd = [np.inf, -np.inf, np.nan, 1e37 if act == "TANH" else 3.4e38]  # (times 1 + o, and then 1 - o)
    D.reshape(-1)[rng.choice(D.size, 12, replace=False)] = odd * 3
    x.reshape(-1)[rng.choice(x.size, 8, replace=False)] = odd[:2] * 4
    y, choice = ctx.empty((rows, C), np.float32), ctx.empty((rows, C), np.int32)
    ctx.maxpool(ctx.array(x), y, d_rules, rows, width, C, choice)
    inverse, samples = ctx.empty((inRows, slots), np.int32), ctx.empty(2 * batch + 1, np.int32)
    ctx.pool_inverse_many([(h, p, d_rules, inverse, samples, rows, inRows, size, stride)])
    background, convInverse = ctx.empty(inRows + 2 * batch, np.int32), ctx.empty((n, fs), np.int32)
    ctx.rules_inverse_many([(g, d_conv, convInverse, background, None, inRows, n, fs)])
    din = ctx.array(np.full((inRows + batch * fs, C), 7, np.float32))
    print("pool gradient not finite", d, field, size, C, act, flush=True)
    ctx.maxpool_gradient(din, inRows, ctx.array(D), rows, C, choice, y if act else None, getattr(scn, act) if act else scn.NOSIGMOID,
                         inverse, slots, samples, batch, background, fs)
    got, ch, v, o = din.download(), choice.download().astype(np.int64), D.astype(np.float64), y.download().astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        if act == "RELU":
            v = np.where(o > 0, v, 0)
        elif act == "LEAKYRELU":
            v = np.where(o > 0, v, v * 0.01)
        elif act == "TANH":
            v = v * ((1 + o) * (1 - o))
        want, size_of = np.zeros((inRows + batch * fs, C)), np.zeros((inRows + batch * fs, C))
        first, mask = samples.download()[:batch + 1], background.download()[:inRows]
        for w, c in zip(*np.nonzero(ch >= 0)):
            r = ch[w, c] // C
            s = np.searchsorted(first, w, side="right") - 1
            for to in [r] + [inRows + s * fs + f for f in range(fs) if mask[r] >> f & 1]:
                want[to, c] += v[w, c]
                size_of[to, c] += abs(v[w, c])
    sure = np.isfinite(want) & (size_of < 3e38)
    assert sure.mean() > 0.9 and not sure.all()
    assert np.all(np.abs(got[sure] - want[sure]) <= 4e-6 * size_of[sure] + 1e-30)
    sure |= size_of > 3e38  # (a sum near the type's largest may round either way)
    sure[~np.isfinite(want)] = False
    assert np.array_equal(np.isnan(got[~sure]), np.isnan(want[~sure])) and np.array_equal(got[~sure], want[~sure].astype(np.float32), equal_nan=True)
