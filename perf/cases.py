"""The work that is timed: what a program built on this framework has it do, through its public entry points.

Six kinds of work, each over its range of sizes:

  net       one batch through a whole net, from the active sites and features in GPU memory to the class
            probabilities on the host (grids, rule books and every layer): an interactive or serving call
  stream    a test pass: batches in turn through the batch producers and the forward lanes
  train     a training epoch over pictures in host memory, and the trained state read back as a checkpoint needs it
  layer     the forward kernels of one layer (convolution, bias, activation, max-pooling) on a batch whose rule
            books stand: a program that drives the C interface with its own containers
  backward  the backward kernels of such a layer
  rules     the rule books of a convolution and of the pooling behind it, from the active sites

A case is a dict of plain values; see listed() for what each listed one stands for.
"""
import functools
import math

import numpy as np
import torch

from __graft_entry__ import load_package

scn = load_package()
from sparseconvnet_archived_amd import hostapi, synthetic  # noqa: E402

PRECISION = {"fp32": scn.FP32, "bf16": scn.BF16}
STACK = {"2d": 2, "3d": 3, "wide": 4}  # the synthetic configurations that end in a classifier
PRODUCERS = 10
LEARNING_RATE = 1e-6  # the last epochs of a schedule


# --------------------------------------------------------------------- cases
def listed():
    return [
        # one character or drawing to be recognised while someone waits: the smallest call
        dict(name="one_drawing", kind="net", stack="2d", batch=1, precision="fp32", fused=True),
        # the batch of the reference's drivers (100 drawings) through the 2-D net
        dict(name="batch_2d", kind="net", stack="2d", batch=100, precision="fp32", fused=True),
        # the same net over a test set, as bench.py runs it
        dict(name="test_pass_2d", kind="stream", stack="2d", batch=100, batches=24),
        # voxelised meshes, an odd last batch, the options as they are by default
        dict(name="batch_3d_default", kind="net", stack="3d", batch=33, precision="fp32", fused=False),
        # a wide net on images, full batch, bf16 operands
        dict(name="batch_wide_bf16", kind="net", stack="wide", batch=128, precision="bf16", fused=True),
        # the same net in fp32 on an odd batch
        dict(name="batch_wide", kind="net", stack="wide", batch=61, precision="fp32", fused=True),
        # an epoch of the 2-D net
        dict(name="epoch_2d", kind="train", stack="2d", batch=100, batches=12),
        # an epoch of the voxel net
        dict(name="epoch_3d", kind="train", stack="3d", batch=32, batches=12),
        # the long layer of the spatio-temporal net (27 taps over 64 channels), fp32: the largest
        dict(name="layer_spacetime", kind="layer", dimension=3, field=126, samples=40, window=3, nIn=64, nOut=64, pool=2,
             precision="fp32"),
        # a layer of that kind with more channels, bf16 operands
        dict(name="layer_spacetime_bf16", kind="layer", dimension=3, field=94, samples=24, window=3, nIn=96, nOut=128,
             pool=2, precision="bf16"),
        # the backward kernels of a middle layer of a 2-D net
        dict(name="backward_2d", kind="backward", dimension=2, field=66, samples=257, window=2, nIn=96, nOut=128, pool=3),
        # the rule books of a spatio-temporal batch
        dict(name="rules_spacetime", kind="rules", dimension=3, field=128, samples=40, window=3, pool=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _field(field, window, pool):
    """the next field that a window of that side and a stride-2 pooling of that side tile"""
    return field + (field - window + 1 - pool) % 2


def draw(rng):
    kind = rng.choice(["net", "net", "stream", "train", "layer", "layer", "backward", "rules"])
    if kind == "net":
        stack = rng.choice(sorted(STACK))
        return dict(kind=kind, stack=stack, batch=_log(rng, 1, {"2d": 200, "3d": 64, "wide": 128}[stack]),
                    precision=rng.choice(["fp32", "fp32", "bf16"]), fused=rng.random() < 0.7)
    if kind == "stream":
        stack = rng.choice(["2d", "3d"])
        return dict(kind=kind, stack=stack, batch=_log(rng, 8, {"2d": 120, "3d": 40}[stack]), batches=rng.randint(12, 24))
    if kind == "train":
        stack = rng.choice(["2d", "3d"])
        return dict(kind=kind, stack=stack, batch=_log(rng, 8, {"2d": 100, "3d": 32}[stack]), batches=rng.randint(5, 12))
    dimension = rng.choice([2, 3])
    if kind == "rules":
        window = rng.choice([2, 3])
        return dict(kind=kind, dimension=dimension,
                    field=_field(rng.randint(40, 160 if dimension == 2 else 126), window, 2),
                    samples=_log(rng, 2, 256 if dimension == 2 else 40), window=window, pool=2)
    window = rng.choice([2, 3])
    pool = rng.choice([2, 3]) if dimension == 2 else 2
    widest = 10 if dimension == 2 else 4  # learnt layers have multiples of 32 channels
    nIn = 32 * rng.randint(1, widest)
    if kind == "layer" and rng.random() < 0.15:
        nIn = rng.randint(1, 4)  # the first layer of a net
    c = dict(kind=kind, dimension=dimension, field=_field(rng.randint(40, 130 if dimension == 2 else 110), window, pool),
             samples=_log(rng, 2, 256 if dimension == 2 else 40), window=window, nIn=nIn,
             nOut=32 * rng.randint(1, widest), pool=pool)
    if kind == "layer":
        c["precision"] = rng.choice(["fp32", "fp32", "bf16"])
    # (no more than the listed ones take, in arithmetic and in memory)
    most = (4e11, 8e9) if kind == "layer" else (6e10, 2e9)
    while c["samples"] > 1 and (work(c)["flops"] > most[0] or _memory(c) > most[1]):
        c["samples"] = max(1, c["samples"] * 2 // 3)
    return c


# ---------------------------------------------------------- active sites, made from a seed
def _fold(p, size):
    """walks that bounce off the borders of [0, size - 1]"""
    m = 2.0 * (size - 1)
    p = np.mod(p, m)
    return np.minimum(p, m - p)


def _strokes(rng, n, size, target):
    """pen strokes: four walks with momentum a sample, about `target` sites in all -> (sample, coordinates)"""
    steps = max(4, target // 4 + target // 8)
    angle = rng.uniform(0, 2 * np.pi, (n, 4, 1)) + np.cumsum(rng.normal(0, 0.35, (n, 4, steps)), 2)
    start = rng.uniform(0.15 * size, 0.85 * size, (n, 4, 1, 2))
    pos = start + np.cumsum(np.stack([np.cos(angle), np.sin(angle)], 3), 2)
    keep = np.arange(steps) < rng.integers(steps // 2, steps + 1, (n, 4, 1))
    at = np.rint(_fold(pos, size)).astype(np.int64)
    sample = np.broadcast_to(np.arange(n)[:, None, None], keep.shape)
    return sample[keep], at[keep]


def _surfaces(rng, n, size):
    """voxels of closed surfaces (ellipsoids with bumps)"""
    pts = 9000
    u = rng.uniform(0, 2 * np.pi, (n, pts))
    w = np.arccos(rng.uniform(-1, 1, (n, pts)))
    ax = size * rng.uniform(0.17, 0.31, (n, 3))
    bump = 1 + 0.12 * np.sin(3 * u + rng.uniform(0, 6, (n, 1))) * np.sin(2 * w)
    p = np.stack([np.sin(w) * np.cos(u), np.sin(w) * np.sin(u), np.cos(w)], 2) * bump[:, :, None] * ax[:, None, :]
    turn = np.linalg.qr(rng.standard_normal((n, 3, 3)))[0]
    at = np.clip(np.rint(np.matmul(p, turn) + (size - 1) / 2.0), 0, size - 1).astype(np.int64)
    return np.repeat(np.arange(n), pts), at.reshape(-1, 3)


def _blobs(rng, n, size):
    """six discs a sample that move through time (axis 0)"""
    vel = 0.25 * rng.standard_normal((n, 6, size, 2))
    for t in range(1, size):
        vel[:, :, t] += 0.9 * vel[:, :, t - 1]
    pos = 3 + _fold(rng.uniform(0.2 * size, 0.8 * size, (n, 6, 1, 2)) + np.cumsum(vel, 2), size - 6)
    o = np.stack(np.meshgrid(np.arange(-3, 4), np.arange(-3, 4), indexing="ij"), 2).reshape(-1, 2)
    at = np.rint(pos)[:, :, :, None, :] + o
    keep = ((at - pos[:, :, :, None, :]) ** 2).sum(4) <= 4.8
    s, _, t, _ = np.nonzero(keep)
    return s, np.concatenate([t[:, None], at[keep].astype(np.int64)], 1)


def _pattern(rng, what, n, size):
    if what == "2d":
        return _strokes(rng, n, size, 4 * size)
    if what == "3d":
        return _surfaces(rng, n, size)
    if what == "wide":
        block = synthetic.dense_block(size, 32).astype(np.int64)
        return np.repeat(np.arange(n), len(block)), np.tile(block, (n, 1))
    return _blobs(rng, n, size)


def _codify(rng, what, n, lattice, field):
    """The active sites of n samples as Picture::codifyInputData leaves them: per sample a background row, then a
    row for every site in order of first appearance -> sample, key, row, background, number of rows."""
    sample, at = _pattern(rng, what, n, lattice)
    shift = (field - lattice) // 2
    key = np.zeros(len(sample), np.int64)
    for a in range(at.shape[1]):
        key = key * field + at[:, a] + shift
    volume = field ** at.shape[1]
    first = np.sort(np.unique(sample * volume + key, return_index=True)[1])
    sample = sample[first].astype(np.int32)
    return (sample,) + _rows(sample, key[first], n)


def _rows(sample, key, n):
    """-> key, row, background, number of rows"""
    row = np.arange(len(key), dtype=np.int64) + sample + 1
    background = np.concatenate([[0], np.cumsum(np.bincount(sample, minlength=n))[:-1]]) + np.arange(n)
    return key.astype(np.int64), row.astype(np.int32), background.astype(np.int32), len(key) + n


class _Buffer:
    """device memory of torch's as the C interface's wrappers take it"""

    def __init__(self, t):
        self.t, self.ptr, self.size = t, t.data_ptr(), t.numel()


def _up(a):
    return _Buffer(torch.from_numpy(np.ascontiguousarray(a)).cuda())


def _room(shape, dtype=torch.float32):
    return _Buffer(torch.empty(shape, dtype=dtype, device="cuda"))


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


# ----------------------------------------------------------------------- nets
def _net(case, threads, seed):
    cfg = synthetic.config(STACK[case["stack"]], batch=case["batch"])
    net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, threads=threads)
    cfg.build(net)
    net.setFusedConvolutions(case.get("fused", case["kind"] != "train"))
    net.setPrecision(PRECISION[case.get("precision", "fp32")])
    rng = np.random.default_rng(seed)
    for i, (W, B, slopes) in synthetic.he_normal_weights(net.layers(), seed).items():
        # (biases as training leaves them: a background row does not sit on the threshold of its rectifier)
        net.set_weights(i, W, 0.05 * rng.standard_normal(B.shape, dtype=np.float32), slopes)
    return cfg, net


def _inputs(rng, cfg, what, batch, field):
    """a batch in GPU memory: (batch, sample, key, row, background, nActive, nSpatialSites, features)"""
    sample, key, row, background, n = _codify(rng, what, batch, cfg.lattice, field)
    feats = np.ones((n, 1), np.float32) if what == "3d" else rng.standard_normal((n, cfg.nInputFeatures), dtype=np.float32)
    feats[background] = 0
    return [batch, _up(sample), _up(key), _up(row), _up(background), len(key), n, _up(feats)]


def _pointers(batch):
    return tuple(x.ptr if isinstance(x, _Buffer) else x for x in batch)


def _prepare_net(case, seed):
    rng = np.random.default_rng(seed)
    cfg, net = _net(case, 1, seed)
    return dict(net=net, inputs=_inputs(rng, cfg, case["stack"], case["batch"], net.inputSpatialSize),
                probs=np.zeros((case["batch"], cfg.nClasses), np.float32))


def _run_net(s):
    s["net"].forward_resident(*_pointers(s["inputs"]), h_probs=s["probs"])
    return s["probs"]


def _prepare_stream(case, seed):
    rng = np.random.default_rng(seed)
    cfg, net = _net(case, PRODUCERS, seed)
    # (two producer streams where the forward pass is the longer half, all of them where the rule books are)
    net.setProducerStreams(2 if case["stack"] == "2d" else 0)
    batches = [_inputs(rng, cfg, case["stack"], case["batch"], net.inputSpatialSize) for _ in range(6)]
    probs = np.zeros((case["batches"], case["batch"], cfg.nClasses), np.float32)
    net.collect_probabilities(probs)
    return dict(net=net, inputs=batches, n=case["batches"], probs=probs)


def _run_stream(s):
    s["net"].forward_stream_timed_many(0, s["n"], [_pointers(b) for b in s["inputs"]])
    return s["probs"]


def _prepare_train(case, seed):
    rng = np.random.default_rng(seed)
    cfg, net = _net(case, PRODUCERS, seed)
    net.set_training(LEARNING_RATE, 0.9, shuffle=False)
    ds = hostapi.Dataset("epoch", cfg.nInputFeatures, cfg.nClasses, hostapi.TRAINBATCH)
    pictures = case["batch"] * case["batches"]
    sample, key, _, _, _ = _codify(rng, case["stack"], pictures, cfg.lattice, cfg.lattice)
    coords = np.stack(np.unravel_index(key, (cfg.lattice,) * cfg.dimension), 1).astype(np.int32)
    feats = (np.ones((len(key), 1), np.float32) if case["stack"] == "3d"
             else rng.standard_normal((len(key), cfg.nInputFeatures), dtype=np.float32))
    ends = np.cumsum(np.bincount(sample, minlength=pictures))
    labels = rng.integers(0, cfg.nClasses, pictures)
    for i, end in enumerate(ends):
        begin = ends[i - 1] if i else 0
        ds.add_points(cfg.dimension, cfg.lattice, coords[begin:end], feats[begin:end], int(labels[i]))
    return dict(net=net, ds=ds, batch=case["batch"], learnt=[i for i, l in enumerate(net.layers()) if l["kind"].startswith("nin")])


def _run_train(s):
    s["net"].processDatasetTrain(s["ds"], s["batch"], LEARNING_RATE, 0.9)
    return [s["net"].get_weights(i, momentum) for i in s["learnt"] for momentum in (False, True)]


# ---------------------------------------------------------------- one layer
def _what(case):
    return "2d" if case["dimension"] == 2 else "blobs"


def _one_layer_sites(case, seed):
    """The sites of a layer's samples.  A seed mirrors, turns and reorders the samples of its own: other sites, as
    many of them at every depth (windows tile the field alike from both ends)."""
    f, d, n = case["field"], case["dimension"], case["samples"]
    sample, key, _, _, _ = _codify(np.random.default_rng(2015), _what(case), n, f, f)
    rng = np.random.default_rng(seed)
    at = np.stack(np.unravel_index(key, (f,) * d), 1)
    at = np.where(rng.integers(0, 2, (n, d))[sample] == 1, f - 1 - at, at)
    swapped = rng.integers(0, 2, n)[sample] == 1
    at[swapped, d - 2], at[swapped, d - 1] = at[swapped, d - 1], at[swapped, d - 2]
    sample = rng.permutation(n)[sample]
    order = np.argsort(sample, kind="stable")
    sample, key = sample[order].astype(np.int32), np.ravel_multi_index(tuple(at[order].T), (f,) * d)
    return (sample,) + _rows(sample, key, n)


def _prepare_sites(case, seed):
    ctx = scn.Context()
    sample, key, row, background, n = _one_layer_sites(case, seed)
    return ctx, [_up(a) for a in (sample, key, row, background)], len(key), n


def _prepare_rules(case, seed):
    ctx, sites, nActive, n = _prepare_sites(case, seed)
    s = dict(case, ctx=ctx, sites=sites, nActive=nActive, rows=n, grids=[scn.Grids(ctx) for _ in range(3)])
    _, sizes = _plan(s)
    s["rules"] = [_room(int(1.2 * k) + 64, torch.int32) for k in sizes]  # the buffers that a program keeps
    return s


def _plan(s, fill=False):
    """input grids, the convolution's rule book, the pooling's -> rows and rules of both"""
    g, f = s["grids"], s["field"]
    f1 = f - s["window"] + 1
    f2 = (f1 - s["pool"]) // 2 + 1
    d = s["dimension"]
    g[0].build_device(s["samples"], d, f, *s["sites"], s["nActive"], s["rows"])
    n1 = g[0].plan_square(g[1], f, f1, s["window"], 1)
    k1 = n1 * s["window"] ** d
    if fill:
        g[0].fill(g[1], s["rules"][0], k1)
    n2 = g[1].plan_square(g[2], f1, f2, s["pool"], 2)
    k2 = n2 * s["pool"] ** d
    if fill:
        g[1].fill(g[2], s["rules"][1], k2)
    return (n1, n2), (k1, k2)


def _run_rules(s):
    rows, sizes = _plan(s, fill=True)
    return [r.t[:k] for r, k in zip(s["rules"], sizes)] + list(rows)


def _prepare_layer(case, seed):
    s = _prepare_rules(case, seed)
    (s["n1"], s["n2"]), _ = _plan(s, fill=True)
    s["ctx"].sync()
    gen = torch.Generator("cuda").manual_seed(seed)
    s["fs"] = fs = case["window"] ** case["dimension"]
    K, N = fs * case["nIn"], case["nOut"]
    # activations as a rectified layer leaves them; the raw values of a first layer
    x = _normal(gen, s["rows"], case["nIn"])
    s["x"] = _Buffer(torch.relu(x) if case["nIn"] >= 32 else x)
    s["W"] = _Buffer(_normal(gen, K, N) * math.sqrt(2.0 / K))
    s["B"] = _Buffer(0.1 * _normal(gen, N))
    s["y"], s["pooled"] = _room((s["n1"], N)), _room((s["n2"], N))
    s["choice"] = _room((s["n2"], N), torch.int32)
    s["precision"] = PRECISION[case.get("precision", "fp32")]
    if not scn.lib().scn_conv_nin_supported_p(fs, case["nIn"], N, s["precision"]):
        s["matrix"] = _room((s["n1"], K))
    elif case.get("precision") == "bf16" and case["nIn"] % 8 == 0 and fs >= 8:
        s["x16"] = _room(s["rows"] * case["nIn"], torch.bfloat16)
    return s


def _run_layer(s):
    ctx, fs, nIn, N = s["ctx"], s["fs"], s["nIn"], s["nOut"]
    if "matrix" in s:
        ctx.gather_rows(s["x"], s["matrix"], s["rules"][0], s["n1"] * fs, nIn)
        ctx.nin_forward(s["matrix"], s["W"], s["B"], None, s["y"], s["n1"], fs * nIn, N, precision=s["precision"])
    elif "x16" in s:
        ctx.conv_nin_forward_a16(s["x"], s["rows"], s["x16"], s["rules"][0], fs, nIn, s["W"], s["B"], None, s["y"],
                                 s["n1"], N)
    else:
        ctx.conv_nin_forward(s["x"], s["rules"][0], fs, nIn, s["W"], s["B"], None, s["y"], s["n1"], N,
                             precision=s["precision"])
    ctx.maxpool(s["y"], s["pooled"], s["rules"][1], s["n2"], s["pool"] ** s["dimension"], N, s["choice"])
    return [s["y"].t, s["pooled"].t, s["choice"].t]


def _prepare_backward(case, seed):
    s = _prepare_layer(case, seed)
    fs, K, N = s["fs"], s["fs"] * case["nIn"], case["nOut"]
    s.pop("matrix", None)
    s["matrix"] = _room((s["n1"], K))  # the gathered matrix that the forward pass of a training batch leaves
    torch.cuda.synchronize()
    _run_layer(s)
    s["ctx"].sync()
    gen = torch.Generator("cuda").manual_seed(seed + 1)
    s["dPooled"] = _Buffer(0.01 * _normal(gen, s["n2"], N))
    s["dy"], s["dMatrix"], s["dx"] = _room((s["n1"], N)), _room((s["n1"], K)), _room((s["rows"], case["nIn"]))
    s["dW"], s["dB"] = _room((K, N)), _room(N)
    s["workspace"] = _room(int(scn.lib().scn_sgemm_ABt_workspace(N, K)))
    return s


def _run_backward(s):
    ctx, fs, nIn, N = s["ctx"], s["fs"], s["nIn"], s["nOut"]
    K = fs * nIn
    scn.lib().scn_fill32(ctx.h, s["dy"].ptr, 0, s["dy"].size)
    ctx.maxpool_backward(s["dy"], s["dPooled"], s["n2"], N, s["choice"])
    ctx.activation_backward(s["y"], s["dy"], s["n1"], N, scn.RELU, None, s["dB"], None)
    ctx.sgemm_AtB(s["matrix"], s["dy"], s["dW"], s["n1"], K, N)
    ctx.sgemm_ABt(s["dy"], s["W"], s["dMatrix"], s["n1"], N, K, s["workspace"])
    scn.lib().scn_fill32(ctx.h, s["dx"].ptr, 0, s["dx"].size)
    ctx.gather_rows_backward(s["dx"], s["dMatrix"], s["rules"][0], s["n1"] * fs, nIn)
    return [s["dW"].t, s["dB"].t, s["dx"].t]


_PREPARE = dict(net=_prepare_net, stream=_prepare_stream, train=_prepare_train, layer=_prepare_layer,
                backward=_prepare_backward, rules=_prepare_rules)
_RUN = dict(net=_run_net, stream=_run_stream, train=_run_train, layer=_run_layer, backward=_run_backward,
            rules=_run_rules)


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, seed), run=_RUN[case["kind"]])


def run(state):
    return state["run"](state)


# ------------------------------------------------------- work and tolerance
@functools.lru_cache(maxsize=None)
def _sites_per_sample(what, lattice, field, dimension, windows):
    """active sites of a typical sample at every depth of a chain of (side, stride) windows"""
    counts = []
    for seed in (0, 1):
        _, key, _, _, _ = _codify(np.random.default_rng(seed), what, 1, lattice, field)
        mask = np.zeros((field,) * dimension, bool)
        mask.reshape(-1)[key] = True
        c = [int(mask.sum())]
        for side, stride in windows:
            n = (mask.shape[0] - side) // stride + 1
            for axis in range(dimension):
                take = lambda o: np.take(mask, np.arange(n) * stride + o, axis)  # noqa: B023, E731
                mask = functools.reduce(np.logical_or, [take(o) for o in range(side)])
            c.append(int(mask.sum()))
        counts.append(c)
    return tuple(sum(x) / len(counts) for x in zip(*counts))


def _layer_sizes(case):
    windows = ((case["window"], 1), (case["pool"], 2))
    n = _sites_per_sample(_what(case), case["field"], case["field"], case["dimension"], windows)
    return [case["samples"] * (1 + x) for x in n]


def _memory(case):
    """bytes of a layer's buffers"""
    r0, r1, r2 = _layer_sizes(case)
    K = case["nIn"] * case["window"] ** case["dimension"]
    wide = 2 * K if case["kind"] == "backward" else 0
    return 4 * (r0 * case["nIn"] + r1 * (2 * case["nOut"] + wide + K / case["nIn"]) + 3 * r2 * case["nOut"])


@functools.lru_cache(maxsize=None)
def _net_sizes(stack):
    """(input sites and features, [(rows, K, N)] of the learnt layers, weights) of one sample"""
    cfg = synthetic.config(STACK[stack])
    d, width = cfg.dimension, cfg.nInputFeatures
    windows, learnt, depth = [], [], 0
    for call in cfg.stack:
        if call[0] == "addLeNetLayerMP":
            _, nOut, side, stride, pool, poolStride = call[:6]
            if side > 1:
                windows.append((side, stride))
                width *= side ** d
            learnt.append((len(windows), width, nOut))
            width = nOut
            if pool > 1:
                windows.append((pool, poolStride))
        elif call[0] == "addTerminalPoolingLayer":
            field = call[1]
    learnt.append((-1, width, cfg.nClasses))
    for side, stride in reversed(windows):
        field = (field - 1) * stride + side
    n = _sites_per_sample(stack, cfg.lattice, field, d, tuple(windows))
    rows = [(1 + n[at] if at >= 0 else 1, K, N) for at, K, N in learnt]
    return n[0], cfg.nInputFeatures, rows, sum((K + 1) * N for _, K, N in learnt), cfg.nClasses


def work(case):
    kind = case["kind"]
    if kind in ("net", "stream", "train"):
        sites, nIn, rows, weights, nClasses = _net_sizes(case["stack"])
        samples = case["batch"] * case.get("batches", 1)
        macs = [m * K * N for m, K, N in rows]
        byts = samples * (sites * 16 + (1 + sites) * 4 * nIn + 4 * nClasses) + 4 * weights
        if kind == "train":  # forward, dW, and d input of every layer but the first; weights and momentum read and written
            return dict(bytes=byts + 12 * weights, flops=2 * samples * (3 * sum(macs) - macs[0]))
        return dict(bytes=byts, flops=2 * samples * sum(macs))
    r0, r1, r2 = _layer_sizes(case)
    fs, ps = case["window"] ** case["dimension"], case["pool"] ** case["dimension"]
    if kind == "rules":
        return dict(bytes=16 * r0 + 4 * (fs * r1 + ps * r2), flops=0)
    nIn, N = case["nIn"], case["nOut"]
    K = fs * nIn
    if kind == "layer":
        return dict(bytes=4 * (r0 * nIn + fs * r1 + K * N + N + r1 * N + ps * r2 + 2 * r2 * N), flops=2 * r1 * K * N)
    return dict(bytes=4 * (2 * r2 * N + r1 * N + r1 * K + 2 * K * N + N + fs * r1 + r0 * nIn), flops=4 * r1 * K * N)


def tolerance(case):
    kind = case["kind"]
    if kind == "rules":
        return "exact"
    # (whole values: a pooling whose two largest inputs are a rounding apart)
    if case.get("precision") == "bf16":
        return {"rel": 1e-2, "differ": 5e-3}
    if kind == "train":
        # one rectifier of millions that a rounding puts on the other side of its threshold takes its share of the
        # gradient with it; a background row's share, common to many sites, is some 1e-3
        return {"rel": 2e-3}
    return {"rel": 1e-5, "differ": 1e-3}
