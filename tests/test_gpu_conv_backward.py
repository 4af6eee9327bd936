"""The backward pass of a convolution without its gathered matrix: dW through the rules, and the input's gradient as a
convolution of the output's through the rules turned round, background rows included; then whole epochs, in which the
host classes take that way, against the net-level oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle_net
from test_gpu_training import pair, rel_l2

pytestmark = pytest.mark.gpu


def layer(scn, ctx, d, field, window, batch, density, seed, stride=1):
    """input grids, their rows, the rules of a convolution [rows x window^d]; sample 1 has no site, sample 2 is full"""
    rng = np.random.default_rng(seed)
    vol = field ** d
    S, K, R, bg, n = [], [], [], [], 0
    for s in range(batch):
        keys = np.nonzero(rng.random(vol) < density)[0] if s != 2 else np.arange(vol)
        keys = keys[:0] if s == 1 else keys
        full = len(keys) == vol
        bg.append(-1 if full else n + len(keys))
        S += [s] * len(keys)
        K += list(keys)
        R += list(range(n, n + len(keys)))
        n += len(keys) + (not full)
    g, h = scn.Grids(ctx), scn.Grids(ctx)
    g.build(batch, d, field, np.array(S, np.int32), np.array(K, np.int64), np.array(R, np.int32), np.array(bg, np.int32), n)
    out = (field - window) // stride + 1
    rows = g.plan_square(h, field, out, window, stride)
    fs = window ** d
    rules = ctx.empty((rows, fs), np.int32)
    g.fill(h, rules, rows * fs)
    return g, n, rows, fs, rules, bg


@pytest.mark.parametrize("d,field,window,batch,density,nIn,N,stride", [
    (2, 9, 2, 1, 0.3, 32, 32, 1), (2, 11, 3, 4, 0.2, 32, 36, 1), (3, 6, 2, 5, 0.1, 64, 96, 1), (3, 7, 3, 3, 0.05, 32, 64, 1),
    (2, 40, 2, 30, 0.15, 96, 128, 1), (2, 13, 3, 6, 0.4, 4, 300, 1), (1, 50, 2, 3, 0.2, 32, 32, 1), (2, 12, 2, 5, 0.3, 160, 64, 2),
    (3, 20, 2, 9, 0.02, 32, 64, 1)])
def test_gradients_through_rules(scn, ctx, d, field, window, batch, density, nIn, N, stride):
    rng = np.random.default_rng(field * window + N)
    g, n, rows, fs, d_rules, bg = layer(scn, ctx, d, field, window, batch, density, field + N, stride)
    print("conv backward", d, field, window, batch, nIn, N, "rows", rows, "of", n, flush=True)
    rules = d_rules.download()
    x, D = rng.standard_normal((n, nIn), dtype=np.float32), rng.standard_normal((rows, N), dtype=np.float32)
    W = rng.standard_normal((fs * nIn, N), dtype=np.float32)
    d_x, d_W = ctx.array(x), ctx.array(W)
    # the rules turned round
    inverse = ctx.array(np.full((n, fs), 7, np.int32))
    pitch = (rows + 15) // 16 * 16
    background, positions = ctx.array(np.full(rows + 2 * batch, 7, np.int32)), ctx.array(np.full((fs, pitch), 7, np.int32))
    ctx.rules_inverse_many([(g, d_rules, inverse, background, positions, rows, n, fs)])
    want = np.full((n, fs), -1, np.int64)
    for s, b in enumerate(bg):
        if b >= 0:
            want[b] = rows + s * fs + np.arange(fs)
    isBg = np.isin(rules, [b for b in bg if b >= 0])
    o, f = np.nonzero((rules >= 0) & ~isBg)
    want[rules[o, f], f] = o
    assert np.array_equal(inverse.download(), want)
    assert np.array_equal(positions.download(), np.pad(rules.T, ((0, 0), (0, pitch - rows)), constant_values=-1))
    got = background.download()
    assert np.array_equal(got[:rows].astype(np.uint32), (isBg * (1 << np.arange(fs, dtype=np.uint32))).sum(1))
    for s, b in enumerate(bg):
        mine = np.nonzero((rules == b).any(1))[0] if b >= 0 else []
        assert tuple(got[rows + 2 * s:rows + 2 * s + 2]) == ((mine[0], mine[-1]) if len(mine) else (2 ** 31 - 1, -1))
    only = ctx.array(np.full((fs, pitch), 7, np.int32))  # (what a net's first convolution wants)
    ctx.rules_inverse_many([(g, d_rules, None, None, only, rows, n, fs)])
    assert np.array_equal(only.download(), positions.download())
    # dW, from zero and added to
    dense = np.where(rules[:, :, None] >= 0, x[np.maximum(rules, 0)], 0).reshape(rows, fs * nIn).astype(np.float64)
    start = rng.standard_normal(W.shape, dtype=np.float32)
    for add in (False, True):
        dW = ctx.array(start)
        ctx.conv_AtB(d_x, positions, fs, nIn, ctx.array(D), dW, rows, N, accumulate=add)
        scale = np.abs(dense).T @ np.abs(D) + np.abs(start)
        assert np.all(np.abs(dW.download() - add * start - dense.T @ D) <= 2e-6 * scale)
    dW, db = ctx.array(start), ctx.array(start[0])
    ctx.conv_AtB(d_x, positions, fs, nIn, ctx.array(D), dW, rows, N, d_db=db)
    assert np.all(np.abs(dW.download() - dense.T @ D) <= 2e-6 * scale)
    assert np.all(np.abs(db.download() - D.astype(np.float64).sum(0)) <= 2e-6 * np.abs(D).astype(np.float64).sum(0))
    # the input's gradient
    Wt = ctx.array(np.full(W.size, 7, np.float32))
    ctx.transpose_filters_many([(d_W, Wt, fs, nIn, N)])
    assert np.array_equal(Wt.download().reshape(fs, N, nIn), W.reshape(fs, nIn, N).transpose(0, 2, 1))
    delta = ctx.array(np.concatenate([D, np.zeros((batch * fs, N), np.float32)]))
    ctx.background_sums(delta, rows, N, background, fs, batch)
    got = delta.download()
    assert np.array_equal(got[:rows], D)
    sums, size = np.zeros((batch * fs, N)), np.zeros((batch * fs, N))
    for s, b in enumerate(bg):
        for q in range(fs):
            sums[s * fs + q] = D[rules[:, q] == b].astype(np.float64).sum(0) if b >= 0 else 0
            size[s * fs + q] = np.abs(D[rules[:, q] == b]).astype(np.float64).sum(0) if b >= 0 else 0
    assert np.all(np.abs(got[rows:] - sums) <= 2e-6 * size)
    dx = ctx.array(np.full((n, nIn), 7, np.float32))
    ctx.conv_input_gradient(delta, inverse, fs, N, Wt, dx, n, nIn)
    want, size = np.zeros((n, nIn)), np.zeros((n, nIn))
    o, f = np.nonzero(rules >= 0)
    dA = (D.astype(np.float64) @ W.astype(np.float64).T).reshape(rows, fs, nIn)
    absA = (np.abs(D).astype(np.float64) @ np.abs(W).astype(np.float64).T).reshape(rows, fs, nIn)
    np.add.at(want, rules[o, f], dA[o, f])
    np.add.at(size, rules[o, f], absA[o, f])
    assert np.all(np.abs(dx.download() - want) <= 4e-6 * size)


@pytest.mark.parametrize("d,field,window,batch,density,nIn,N", [(2, 110, 2, 12, 0.15, 64, 64), (2, 110, 2, 12, 0.15, 96, 64)])
def test_gradient_with_the_filters_laid_out(scn, ctx, d, field, window, batch, density, nIn, N):
    """as epochs have it: through inverse rules, the rows of sums behind delta's own among them, the bits without"""
    rng = np.random.default_rng(field)
    g, n, rows, fs, d_rules, bg = layer(scn, ctx, d, field, window, batch, density, field + N)
    print("turned image", d, field, window, nIn, N, "rows", rows, "of", n, flush=True)
    d_W = ctx.array(rng.standard_normal((fs * nIn, N), dtype=np.float32))
    delta = ctx.array(np.concatenate([rng.standard_normal((rows, N), dtype=np.float32), np.zeros((batch * fs, N), np.float32)]))
    inverse, background, Wt = ctx.empty((n, fs), np.int32), ctx.empty(rows + 2 * batch, np.int32), ctx.empty(fs * nIn * N, np.float32)
    ctx.rules_inverse_many([(g, d_rules, inverse, background, None, rows, n, fs)])
    assert (inverse.download() >= rows).any()
    ctx.background_sums(delta, rows, N, background, fs, batch)
    ctx.transpose_filters_many([(d_W, Wt, fs, nIn, N)])
    size = scn.lib().scn_weight_image_bytes(ctx.h, n, fs * N, nIn, N, scn.FP32_PLANES)
    assert size > 0
    image, outs = ctx.empty(size // 4, np.float32), [ctx.array(np.full((n, nIn), 7, np.float32)) for _ in range(2)]
    ctx.weight_images_many([(d_W, image, fs * N, nIn, fs, scn.FP32_PLANES)])
    for out, im in zip(outs, (None, image)):
        ctx.conv_input_gradient(delta, inverse, fs, N, Wt, out, n, nIn, d_image=im)
    assert np.array_equal(outs[0].download(), outs[1].download())


# all layers' weight gradients in one launch: rows through rules by lines (whole tiles and not), a first layer's of three
# channels, plain rows; no rows, fewer than a step, more than a workgroup's share; a shape that goes by itself (N 31); more
# tiles than compute units (1600 x 512: 400) beside others
@pytest.mark.parametrize("plain", [[(1, 32, 32)], [(100, 160, 192), (0, 32, 32), (100, 192, 100), (130, 34, 31)],
                                   [(5000, 1600, 512), (33, 64, 4), (20001, 96, 128)]])
@pytest.mark.parametrize("convs", [[], [(2, 11, 3, 4, 0.2, 32, 36), (2, 40, 2, 9, 0.15, 3, 32), (3, 7, 3, 3, 0.05, 64, 64)],
                                   [(2, 60, 2, 40, 0.15, 36, 64), (1, 50, 2, 3, 0.2, 32, 32)]])
def test_weight_gradients_of_many_layers(scn, ctx, plain, convs):
    rng = np.random.default_rng(len(plain) + 7 * len(convs))
    items, checks = [], []
    for M, K, N in plain:
        A, D = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((M, N), dtype=np.float32)
        items.append((ctx.array(A) if M else None, None, 1, K, ctx.array(D) if M else ctx.empty(1, np.float32), M, N))
        checks.append((A, D))
    for d, field, window, batch, density, nIn, N in convs:
        g, n, rows, fs, d_rules, bg = layer(scn, ctx, d, field, window, batch, density, field + N)
        positions = ctx.empty((fs, (rows + 15) // 16 * 16), np.int32)
        ctx.rules_inverse_many([(g, d_rules, None, None, positions, rows, n, fs)])
        rules = d_rules.download()
        x, D = rng.standard_normal((n, nIn), dtype=np.float32), rng.standard_normal((rows, N), dtype=np.float32)
        items.append((ctx.array(x), positions, fs, nIn, ctx.array(D), rows, N))
        checks.append((np.where(rules[:, :, None] >= 0, x[np.maximum(rules, 0)], 0).reshape(rows, fs * nIn), D))
    print("weight gradients of", [(i[2], i[3], i[5], i[6]) for i in items], flush=True)
    starts = [rng.standard_normal((A.shape[1] + 1, D.shape[1]), dtype=np.float32) for A, D in checks]
    out = [(ctx.array(s[:-1]), ctx.array(s[-1]) if k % 3 else None) for k, s in enumerate(starts)]
    ctx.AtB_many([(x, p, fs, nIn, D, dW, db, M, N) for (x, p, fs, nIn, D, M, N), (dW, db) in zip(items, out)])
    for (A, D), s, (dW, db) in zip(checks, starts, out):
        A, D = A.astype(np.float64), D.astype(np.float64)
        assert np.all(np.abs(dW.download() - s[:-1] - A.T @ D) <= 2e-6 * (np.abs(A).T @ np.abs(D) + np.abs(s[:-1])))
        if db is not None:
            assert np.all(np.abs(db.download() - s[-1] - D.sum(0)) <= 2e-6 * (np.abs(D).sum(0) + np.abs(s[-1])))


# every tile that sums take; ragged rows and columns; added to and not
@pytest.mark.parametrize("M,K,N", [(1, 32, 32), (130, 34, 31), (1000, 66, 100), (40001, 12, 32), (30011, 256, 96), (70003, 432, 128),
                                   (53327, 644, 324)])
def test_weight_and_bias_gradients_in_one(scn, ctx, M, K, N):
    rng = np.random.default_rng(M + K + N)
    A, D = rng.standard_normal((M, K), dtype=np.float32), rng.standard_normal((M, N), dtype=np.float32)
    start = rng.standard_normal((K + 1, N), dtype=np.float32)
    print("products with sums", M, K, N, flush=True)
    for add in (False, True):
        dW, db = ctx.array(start[:K]), ctx.array(start[K])
        ctx.sgemm_AtB_sums(ctx.array(A), ctx.array(D), dW, db, M, K, N, accumulate=add)
        scale = np.abs(A).astype(np.float64).T @ np.abs(D).astype(np.float64) + np.abs(start[:K])
        assert np.all(np.abs(dW.download() - add * start[:K] - A.astype(np.float64).T @ D) <= 2e-6 * scale)
        size = np.abs(D).astype(np.float64).sum(0) + np.abs(start[K])
        assert np.all(np.abs(db.download() - add * start[K] - D.astype(np.float64).sum(0)) <= 2e-6 * size)


@pytest.mark.parametrize("n,C", [(1, 4), (2001, 32), (9000, 3), (20000, 96)])
@pytest.mark.parametrize("act", ["NOSIGMOID", "RELU", "VLEAKYRELU", "LEAKYRELU", "TANH", "SIGMOID"])
def test_pooling_gradient_takes_the_derivative(scn, ctx, n, C, act):
    rng = np.random.default_rng(n + C)
    a = getattr(scn, act)
    out = rng.uniform(-1, 1, (n, C)).astype(np.float32)
    out[rng.random((n, C)) < 0.3] = 0
    g = rng.standard_normal((n, C)).astype(np.float32)
    choice = ctx.array((rng.integers(0, 700, (n, C)) * C + np.arange(C)).astype(np.int32))
    dB = ctx.array(np.zeros(C, np.float32))
    two, one = (ctx.array(np.zeros((700, C), np.float32)) for _ in range(2))
    d = ctx.array(g)
    ctx.activation_backward(ctx.array(out), d, n, C, a, None, dB, None)
    ctx.maxpool_backward(two, d, n, C, choice)
    ctx.maxpool_backward_through(one, ctx.array(g), n, C, choice, ctx.array(out), a)
    # (the same products, added in another order)
    size = np.zeros(700 * C)
    np.add.at(size, choice.download().ravel(), np.abs(g).ravel().astype(np.float64))
    assert np.all(np.abs(one.download().ravel() - two.download().ravel()) <= 1e-6 * size)


def test_many_layers_in_one_call(scn, ctx):
    layers = [layer(scn, ctx, 2, 8 + 3 * k, 2 + k % 2, 1 + k, 0.3, k) for k in range(6)]
    one = [ctx.array(np.full((n, fs), 7, np.int32)) for _, n, _, fs, _, _ in layers]
    many = [ctx.array(np.full((n, fs), 7, np.int32)) for _, n, _, fs, _, _ in layers]
    items = [[(g, rules, inv, None, None, rows, n, fs) for (g, n, rows, fs, rules, _), inv in zip(layers, to)] for to in (one, many)]
    for it in items[0]:
        ctx.rules_inverse_many([it])
    ctx.rules_inverse_many(items[1])
    for a, b in zip(one, many):
        assert np.array_equal(a.download(), b.download())


def test_an_input_without_rows(scn, ctx):
    """rows that name nothing: every sample's first and last row with a background are "none", alone and beside a layer
    that has an inverse; its sums add nothing"""
    g, n, rows, fs, rules, _ = layer(scn, ctx, 2, 8, 2, 3, 0.3, 1)
    batch, N = 3, 8
    none = ctx.array(np.full((rows, fs), -1, np.int32))
    inverse = ctx.array(np.full((n, fs), 7, np.int32))
    for beside in (False, True):
        background, other = (ctx.array(np.full(rows + 2 * batch, 7, np.int32)) for _ in range(2))
        items = [(g, none, inverse, background, None, rows, 0, fs)]
        ctx.rules_inverse_many(items + [(g, rules, inverse, other, None, rows, n, fs)] * beside)
        got = background.download()
        assert np.all(got[:rows] == 0)
        # (only then may they be taken for rows: a kernel walks from the first to the last)
        assert np.array_equal(got[rows:], np.tile(np.array([2 ** 31 - 1, -1], np.int32), batch))
        delta = np.zeros((rows + batch * fs, N), np.float32)
        delta[:rows] = 1
        d_delta = ctx.array(delta)
        ctx.background_sums(d_delta, rows, N, background, fs, batch)
        assert np.array_equal(d_delta.download(), delta)


def test_refusals(scn, ctx):
    g, n, rows, fs, rules, _ = layer(scn, ctx, 2, 8, 2, 2, 0.3, 1)
    buf = ctx.empty((64, 64), np.float32)
    with pytest.raises(scn.ScnError):
        ctx.conv_AtB(buf, rules, 0, 32, buf, buf, 4, 4)
    with pytest.raises(scn.ScnError):
        ctx.conv_AtB(buf, rules, 4, 5000, buf, buf, 4, 4)  # more channels than the zero row has
    with pytest.raises(scn.ScnError):
        ctx.rules_inverse_many([(g, rules, rules, None, None, rows, n, fs)] * 17)
    with pytest.raises(scn.ScnError):
        ctx.background_sums(buf, 4, 0, rules, fs, 2)
    with pytest.raises(scn.ScnError):
        ctx.maxpool_backward_through(buf, buf, 4, 4, rules, buf, scn.PRELU)  # its slopes' gradient needs a pass of its own


STACKS = {
    "tri": (True, [("addLeNetLayerMP", 32, 2, 1, 2, 2, 4), ("addLeNetLayerMP", 64, 2, 1, 2, 2, 1), ("addLeNetLayerMP", 64, 2, 1, 1, 1, 3),
                   ("addTerminalPoolingLayer", 2), ("addSoftmaxLayer",)]),
    # convolutions one behind the other, without a pooling between them; the last one's output is one site a sample
    "unpooled": (False, [("addLeNetLayerMP", 32, 3, 1, 1, 1, 1), ("addLeNetLayerMP", 64, 2, 1, 1, 1, 6),
                         ("addLeNetLayerMP", 32, 2, 1, 3, 2, 1), ("addLeNetLayerMP", 32, 2, 1, 1, 1, 1), ("addSoftmaxLayer",)]),
    # rows enough for weights laid out ahead, forwards and turned round
    "laid out": (False, [("addLeNetLayerMP", 64, 3, 1, 2, 2, 4), ("addLeNetLayerMP", 64, 2, 1, 2, 2, 4),
                         ("addLeNetLayerMP", 64, 3, 1, 2, 2, 4), ("addLeNetLayerMP", 64, 2, 1, 1, 1, 4), ("addSoftmaxLayer",)])}


def laid_out(scn, net, cfg, hostapi, samples):
    """of a batch's convolutions: are there layouts of the weights for one of them forwards, and turned round?"""
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TESTBATCH)
    for pts, f, label in samples:
        ds.add_points(cfg.dimension, cfg.lattice, pts, f, label)
    net.begin(ds, len(samples))
    assert net.next_batch()
    info = [net.interface(i, want_features=False) for i in range(len(net.layers()) + 1)]
    net.end()
    size, layers = scn.lib().scn_weight_image_bytes, net.layers()
    forwards = turned = 0
    ctx = C.c_void_p(net.context_handle())
    for i, l in enumerate(layers[1:], 1):
        if l["kind"].startswith("nin") and layers[i - 1]["kind"] == "conv" and i > 1:
            src, out, N = info[i - 1], info[i + 1], l["nOut"]
            nIn, fs = src["nFeatures"], l["nIn"] // src["nFeatures"]
            forwards = max(forwards, size(ctx, out["nSpatialSites"], l["nIn"], N, nIn, scn.FP32_PLANES))
            turned = max(turned, size(ctx, src["nSpatialSites"], fs * N, nIn, N, scn.FP32_PLANES))
            print("rows", out["nSpatialSites"], "of", src["nSpatialSites"], "layouts", forwards, turned, flush=True)
    return forwards, turned


@pytest.mark.parametrize("what,batch,epochs", [(2, 8, 2), (3, 5, 1), (4, 2, 1), ("tri", 4, 2), ("unpooled", 4, 2),
                                               ("laid out", 100, 1)])
def test_epochs_against_the_oracle(scn, what, batch, epochs):
    from sparseconvnet_archived_amd import hostapi, synthetic
    rng = np.random.default_rng(5)
    if isinstance(what, int):
        cfg = synthetic.config(what, batch=2 * batch + 1)
        samples = synthetic.make_samples(cfg, 41)
        triangular = False
    else:
        triangular, stack = STACKS[what]
        lattice = 30 if what == "laid out" else 12
        cfg = synthetic.Config(what, 2, 3, 10, 2 * batch + 1, lattice, stack)
        cfg.number = 2
        samples = []
        for _ in range(2 * batch + 1):
            pts = np.array([(a, b) for a in range(lattice) for b in range(lattice - (a if triangular else 0))
                            if rng.random() < 0.3], np.int32)
            samples.append((pts, rng.uniform(-1, 1, (len(pts), 3)).astype(np.float32), int(rng.integers(0, 10))))
    pts, f, label = samples[1]
    samples[1] = (pts[:0], f[:0], label)  # a sample without a site
    net, ora = pair(cfg, hostapi, 51, triangular)
    if what == "laid out":
        assert all(laid_out(scn, net, cfg, hostapi, samples[:batch]))
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TRAINBATCH)
    for pts, f, label in samples:
        ds.add_points(cfg.dimension, cfg.lattice, pts, f, label)
    lr, mu = 0.01, 0.9
    net.set_training(lr, mu, shuffle=False)
    for _ in range(epochs):
        net.processDatasetTrain(ds, batch, lr, mu)
        for b in range(0, len(samples), batch):  # (the last batch is not full)
            mine = samples[b:b + batch]
            S, K, R, bg, feats, n = synthetic.codify(mine, cfg.dimension, cfg.lattice, net.inputSpatialSize,
                                                     cfg.nInputFeatures)
            labels = np.array([s[2] for s in mine], np.int32)
            fwd = ora.forward(len(mine), S, K, R, bg, feats, n, labels)
            ora.train_step(fwd, labels, lr, mu)
    for i, l in enumerate(net.layers()):
        if not l["kind"].startswith("nin"):
            continue
        M, W = net.get_weights(i, momentum=True), net.get_weights(i)
        err = [rel_l2(a, b) for a, b in zip(M, ora.momentum[i]) if a is not None]
        print("layer", i, "momentum off by", err, flush=True)
        # (the bar of one batch, a batch's share of rectifiers that a rounding turns among them)
        assert max(err) <= 1e-4 * epochs * 3
        for a, b in zip(W, ora.weights[i]):
            if a is not None:
                assert np.allclose(a, b, rtol=1e-4 * epochs * 3, atol=3e-6 * epochs)
    net.close()


def products(a, b):
    """a @ b by columns of a: infinities and NaN as plain sums of products give them, whatever the library does"""
    with np.errstate(invalid="ignore", over="ignore"):
        out = np.zeros((a.shape[0], b.shape[1]))
        for k in range(a.shape[1]):
            out += a[:, k:k + 1] * b[k]
    return out


# split contraction, tiles of whole lines, tiles of k_nin_planes (channels in fours of a position; few rows to a
# workgroup); few rows, tiles and resident weights on the fp32 MFMA
@pytest.mark.parametrize("d,field,window,batch,density,nIn,N", [
    (2, 7, 2, 4, 0.3, 32, 32), (3, 6, 3, 3, 0.1, 32, 64), (2, 110, 2, 12, 0.15, 32, 64), (2, 120, 2, 24, 0.2, 64, 32),
    (2, 110, 2, 12, 0.15, 64, 24), (2, 9, 2, 3, 0.3, 20, 36), (2, 60, 3, 6, 0.2, 32, 36), (2, 70, 2, 9, 0.2, 64, 36)])
def test_infinite_weights_reach_the_rows_that_are_named(scn, ctx, d, field, window, batch, density, nIn, N):
    """as a product per output row, added through the rules, has it: a filter position that no output row names an input
    row at adds nothing to it, not 0 times its weights"""
    rng = np.random.default_rng(field + N)
    g, n, rows, fs, d_rules, bg = layer(scn, ctx, d, field, window, batch, density, field + nIn)
    print("infinite weights", d, field, window, nIn, N, "rows", rows, "of", n, flush=True)
    # (a sum of 250000 rows of D is below 1: what is finite in 64 bits, 3.4e38 times it included, is so in 32)
    rules, D = d_rules.download(), (1e-4 * rng.standard_normal((rows, N))).astype(np.float32)
    W = rng.standard_normal((fs, nIn, N)).astype(np.float32)
    for value in (np.inf, -np.inf, np.nan, 3.4e38):
        W[rng.integers(0, fs), rng.integers(0, nIn), rng.integers(0, N)] = value
    D[rows // 2, 3], D[rows // 3, 1] = np.inf, np.nan
    pitch = scn.lib().scn_positions_pitch(rows)
    inverse, background = ctx.empty((n, fs), np.int32), ctx.empty(rows + 2 * batch, np.int32)
    positions = ctx.empty((fs, pitch), np.int32)
    ctx.rules_inverse_many([(g, d_rules, inverse, background, positions, rows, n, fs)])
    Wt, delta = ctx.empty(W.size, np.float32), ctx.array(np.concatenate([D, np.zeros((batch * fs, N), np.float32)]))
    ctx.transpose_filters_many([(ctx.array(W.reshape(fs * nIn, N)), Wt, fs, nIn, N)])
    ctx.background_sums(delta, rows, N, background, fs, batch)
    want, size = np.zeros((n, nIn)), np.zeros((n, nIn))
    isBg = np.isin(rules, [b for b in bg if b >= 0])
    with np.errstate(invalid="ignore", over="ignore"):
        for f in range(fs):
            Wf = W[f].T.astype(np.float64)
            own = np.nonzero((rules[:, f] >= 0) & ~isBg[:, f])[0]
            want[rules[own, f]] += products(D[own].astype(np.float64), Wf)
            size[rules[own, f]] += products(np.abs(D[own]).astype(np.float64), np.abs(Wf))
            for b in bg:
                mine = np.nonzero(rules[:, f] == b)[0] if b >= 0 else []
                if len(mine):
                    want[b] += products(D[mine].astype(np.float64).sum(0, keepdims=True), Wf)[0]
                    size[b] += products(np.abs(D[mine]).astype(np.float64).sum(0, keepdims=True), np.abs(Wf))[0]
    outs = [ctx.array(np.full((n, nIn), 7, np.float32)) for _ in range(2)]
    ctx.conv_input_gradient(delta, inverse, fs, N, Wt, outs[0], n, nIn)
    if N % 32 == 0:  # (the weights laid out, as epochs have them: the same bits)
        image = ctx.empty((nIn + 31) // 32 * 32 * fs * N * 6 // 4, np.float32)
        ctx.weight_images_many([(ctx.array(W.reshape(fs * nIn, N)), image, fs * N, nIn, fs, scn.FP32_PLANES)])
        ctx.conv_input_gradient(delta, inverse, fs, N, Wt, outs[1], n, nIn, d_image=image)
        assert np.array_equal(outs[1].download(), outs[0].download(), equal_nan=True)
    got, sure = outs[0].download(), np.isfinite(want)
    assert sure.mean() > 0.5 and not sure.all() and size[sure].max() < 3.4e38
    assert np.array_equal(got[~sure], want[~sure].astype(np.float32), equal_nan=True)
    assert np.all(np.abs(got[sure] - want[sure]) <= 4e-6 * size[sure])


@pytest.mark.parametrize("M,fs,nIn,N", [(391, 3, 36, 44), (2051, 4, 32, 64), (391, 4, 7, 33), (9001, 4, 96, 160)])
def test_infinite_operands_of_the_weight_gradient(scn, ctx, M, fs, nIn, N):
    """through the rules (rows by lines, and not): what the gathered matrix's product has, zero rows included"""
    rng = np.random.default_rng(M + nIn)
    # (the sum of a column of D is below 1 in magnitude: what is finite in 64 bits is so in 32)
    x, D = rng.standard_normal((300, nIn)).astype(np.float32), (0.1 / M * rng.standard_normal((M, N))).astype(np.float32)
    x[3, 5], x[77, 2], x[5, 1], x[8, 0], D[M // 2, 11], D[M // 3, 2] = np.inf, -np.inf, np.nan, 3.4e38, np.inf, np.nan
    rules = rng.integers(-1, 300, (M, fs)).astype(np.int32)
    pitch = scn.lib().scn_positions_pitch(M)
    positions = ctx.array(np.ascontiguousarray(np.pad(rules.T, ((0, 0), (0, pitch - M)), constant_values=-1)))
    print("infinite operands of dW", M, fs, nIn, N, flush=True)
    dense = np.where(rules[:, :, None] >= 0, x[np.maximum(rules, 0)], 0).reshape(M, fs * nIn).astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = np.einsum("mk,mn->kn", dense, D.astype(np.float64))
        size, sums = np.einsum("mk,mn->kn", np.abs(dense), np.abs(D).astype(np.float64)), D.astype(np.float64).sum(0)
    dW, db = ctx.array(np.full((fs * nIn, N), 7, np.float32)), ctx.array(np.full(N, 7, np.float32))
    ctx.conv_AtB(ctx.array(x), positions, fs, nIn, ctx.array(D), dW, M, N, d_db=db)
    got, sure = dW.download(), np.isfinite(want)
    assert np.array_equal(got[~sure], want[~sure].astype(np.float32), equal_nan=True)
    assert np.all(np.abs(got[sure] - want[sure]) <= 2e-6 * size[sure])
    got, sure = db.download(), np.isfinite(sums)
    assert np.array_equal(got[~sure], sums[~sure].astype(np.float32), equal_nan=True)
    assert np.all(np.abs(got[sure] - sums[sure]) <= 2e-6 * np.abs(D).sum(0)[sure])


# the same of several layers in one launch: rows by lines, a first layer's without, plain rows, some of more than one range,
# so that a workgroup takes what is not finite again between tiles that are
def test_infinite_operands_among_many_layers(scn, ctx):
    rng = np.random.default_rng(6)
    items, checks = [], []
    for M, fs, nIn, N in ((391, 3, 36, 44), (20011, 4, 32, 64), (9001, 4, 3, 32), (5003, 1, 160, 96), (700, 1, 64, 100)):
        n = 300 if fs > 1 else M
        x, D = rng.standard_normal((n, nIn)).astype(np.float32), (0.1 / M * rng.standard_normal((M, N))).astype(np.float32)
        x[3, 2], x[77, 2], x[5, 1], x[8, 0], D[M // 2, 11], D[M // 3, 2] = np.inf, -np.inf, np.nan, 3.4e38, np.inf, np.nan
        rules = rng.integers(-1, n, (M, fs)).astype(np.int32) if fs > 1 else np.arange(M, dtype=np.int32)[:, None]
        pitch = scn.lib().scn_positions_pitch(M)
        positions = ctx.array(np.ascontiguousarray(np.pad(rules.T, ((0, 0), (0, pitch - M)), constant_values=-1))) if fs > 1 else None
        dense = np.where(rules[:, :, None] >= 0, x[np.maximum(rules, 0)], 0).reshape(M, fs * nIn).astype(np.float64)
        items.append((ctx.array(x), positions, fs, nIn, ctx.array(D), ctx.array(np.zeros((fs * nIn, N), np.float32)),
                      ctx.array(np.zeros(N, np.float32)), M, N))
        checks.append((dense, D.astype(np.float64)))
    print("infinite operands among many", [i[2:4] + i[7:] for i in items], flush=True)
    ctx.AtB_many(items)
    for (dense, D), item in zip(checks, items):
        with np.errstate(invalid="ignore"):
            want = np.einsum("mk,mn->kn", dense, D)
            size, sums = np.einsum("mk,mn->kn", np.abs(dense), np.abs(D)), D.sum(0)
        for got, want, size in ((item[5].download(), want, size), (item[6].download(), sums, np.abs(D).sum(0))):
            sure = np.isfinite(want)
            assert not sure.all() and sure.any()
            assert np.array_equal(got[~sure], want[~sure].astype(np.float32), equal_nan=True)
            assert np.all(np.abs(got[sure] - want[sure]) <= 2e-6 * size[sure])


def test_an_epoch_with_an_infinite_weight(scn):
    """of a channel that is never above zero, so that the net's outputs are finite: an epoch of one batch leaves what the
    batch by itself, which gathers, leaves"""
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(2, batch=8)
    samples = synthetic.make_samples(cfg, 43)
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TRAINBATCH)
    for pts, f, label in samples:
        ds.add_points(cfg.dimension, cfg.lattice, pts, f, label)
    left = []
    for epoch in (True, False):
        net, _ = pair(cfg, hostapi, 52)
        nin = [i for i, l in enumerate(net.layers()) if l["kind"].startswith("nin")]
        W, B, _ = net.get_weights(nin[0])
        B[5] = -1e6
        net.set_weights(nin[0], W, B)
        W, B, _ = net.get_weights(nin[1])
        W[32 + 5, 2] = np.inf  # (its second position)
        net.set_weights(nin[1], W, B)
        net.set_training(0.01, 0.9, shuffle=False)
        if epoch:
            net.processDatasetTrain(ds, 8, 0.01, 0.9)
        else:
            net.begin(ds, 8)
            while net.next_batch():
                pass
        left.append([a for i in nin for m in (True, False) for a in net.get_weights(i, momentum=m) if a is not None])
        net.close()
    for k, (a, b) in enumerate(zip(*left)):
        sure = np.isfinite(b)
        print("tensor", k, "not finite", int((~sure).sum()), "of", b.size, "off by", rel_l2(a[sure], b[sure]), flush=True)
        assert np.array_equal(a[~sure], b[~sure], equal_nan=True)
        # (the same forward pass, bit for bit, so the same rectifiers: what is left are fp32 sums in other orders)
        assert rel_l2(a[sure], b[sure]) <= 1e-5
