"""Recorded plans (scn_ctx_chain_rules): the rule books of consecutive layers
built together, samples side by side, against the CPU oracle -- bit-exact
rules, counts, grids (table and mask built on demand from the entry lists) --
and against the same calls run one by one."""
import numpy as np
import pytest

import brute
import oracle as orc
from gpu_util import assert_same_grids, flatten_samples, oracle_grids

pytestmark = pytest.mark.gpu


class Stack:
    """A source grids object and one output object per layer, reused across batches as the host classes do."""

    def __init__(self, scn, ctx, d, layers, terminal=True):
        # layers: (kind, size, stride, minActive) from the input side; sizes worked out from the top
        self.scn, self.ctx, self.d, self.layers, self.terminal = scn, ctx, d, layers, terminal
        self.src = scn.Grids(ctx)
        self.outs = [scn.Grids(ctx) for _ in layers]
        self.term = scn.Grids(ctx) if terminal else None

    def sizes(self, top):
        s = [top]
        for kind, size, stride, _ in reversed(self.layers):
            s.append(size + (s[-1] - 1) * stride)
        return s[::-1]

    def oracle(self, samples, sizes):
        og, want = oracle_grids(samples), []
        for (kind, size, stride, mn), nIn, nOut in zip(self.layers, sizes[:-1], sizes[1:]):
            fn = orc.rules_triangular if kind == "tri" else orc.rules_square
            og2, rules, n = fn(og, self.d, nIn, nOut, size, stride, mn)
            want.append((og2, rules, n))
            og = og2
        if self.terminal:
            want.append(orc.rules_terminal(og))
        return want

    def build(self, samples, nSites, n):
        objs = [self.src] + self.outs + ([self.term] if self.terminal else [])
        self.scn.clear_many(self.ctx, objs)
        s, k, r, bg = flatten_samples(samples)
        self.src.build(len(samples), self.d, n, s, k, r, bg, nSites)

    def run(self, samples, sizes):
        got, cur = [], self.src
        for (kind, size, stride, mn), nIn, nOut, out in zip(self.layers, sizes[:-1], sizes[1:], self.outs):
            d2, rules, n, w = self.scn.rules_square(self.ctx, cur, nIn, nOut, size, stride, mn,
                                                    triangular=kind == "tri", out=out)
            got.append((d2, rules, n, w))
            cur = d2
        if self.terminal:
            S = cur.plan_terminal(self.term)
            rules = self.ctx.empty(max(len(samples) * S, 1), np.int32)
            cur.fill(self.term, rules, len(samples) * S)
            got.append((self.term, rules, len(samples), S))
        return got

    def run_chained(self, samples, sizes):
        chains, plans = self.scn.chain_count(self.ctx)
        self.scn.defer_counts(self.ctx, True)
        self.scn.chain_rules(self.ctx, True)
        got = self.run(samples, sizes)
        self.scn.chain_rules(self.ctx, False)
        self.scn.defer_counts(self.ctx, False)
        # every layer joined one chain
        assert self.scn.chain_count(self.ctx) == (chains + 1, plans + len(got))
        return got, self.scn.settle(self.ctx)

    def check(self, got, want, batch):
        regions = got[:-1] if self.terminal else got
        for (dg, rules, _, w), (og, o_rules, o_n) in zip(regions, want):
            assert dg.info()["nSpatialSites"] == o_n
            assert np.array_equal(rules.download()[: o_n * w], o_rules)
            assert_same_grids(dg, og)
        if self.terminal:
            (dg, rules, _, _), (og, o_rules, o_S) = got[-1], want[-1]
            assert dg.rules_width() == o_S
            assert np.array_equal(rules.download()[: batch * o_S], o_rules)
            assert_same_grids(dg, og)


def tri_only(samples, n, d):
    return [(bg, {k: r for k, r in mp.items() if sum(brute.decode(k, n, d)) < n}) for bg, mp in samples]


CASES = [
    # d, layers, top size, densities
    ("c2_mp32_2d", 2, [("sq", 2, 1, 1), ("sq", 3, 2, 1), ("sq", 2, 1, 1), ("sq", 3, 2, 1)], 3),
    ("c3_mp2_2d", 2, [("sq", 3, 1, 1), ("sq", 2, 2, 1), ("sq", 3, 1, 1)], 4),
    ("min2_2d", 2, [("sq", 3, 1, 2), ("sq", 2, 2, 1), ("sq", 2, 1, 3)], 5),
    ("valid_2d", 2, [("sq", 3, 1, -1), ("sq", 3, 1, -1), ("sq", 2, 2, 1)], 4),
    ("c2_mp2_3d", 3, [("sq", 2, 1, 1), ("sq", 2, 2, 1), ("sq", 2, 1, 1), ("sq", 2, 2, 1)], 2),
    ("c3_3d", 3, [("sq", 3, 1, 1), ("sq", 3, 2, 1)], 3),
    ("min_3d", 3, [("sq", 2, 1, 2), ("sq", 3, 2, 1)], 3),
    ("c2_mp3_1d", 1, [("sq", 2, 1, 1), ("sq", 3, 3, 1), ("sq", 5, 2, 1)], 4),
    ("tri_2d", 2, [("tri", 2, 1, 1), ("tri", 3, 2, 1), ("tri", 2, 1, 2)], 3),
    ("tri_3d", 3, [("tri", 2, 1, 1), ("tri", 2, 2, 1)], 3),
    ("size1_2d", 2, [("sq", 1, 1, 1), ("sq", 2, 2, 1)], 6),
]


@pytest.mark.parametrize("name,d,layers,top", CASES, ids=[c[0] for c in CASES])
def test_chained_rule_books(scn, ctx, name, d, layers, top):
    rng = np.random.default_rng(len(name) + 17 * d + top)
    st = Stack(scn, ctx, d, layers)
    sizes = st.sizes(top)
    tri = layers[0][0] == "tri"
    print("chain", name, "sizes", sizes, flush=True)

    def draw(batch, density):
        samples, nSites = brute.random_samples(rng, batch, d, sizes[0], density)
        return (tri_only(samples, sizes[0], d) if tri else samples), nSites

    # the first batch is planned layer by layer (no history to bound a recorded plan with)
    samples, nSites = draw(5, 0.3)
    st.build(samples, nSites, sizes[0])
    st.check(st.run(samples, sizes), st.oracle(samples, sizes), 5)
    # recorded batches of every density that fits the bounds, empty and full samples included
    for batch, density in ((5, 0.25), (4, 0.02), (5, 0.31), (3, 0.0)):
        samples, nSites = draw(batch, density)
        if density > 0.2:
            samples[1] = (samples[1][0], {})  # a sample without sites
        st.build(samples, nSites, sizes[0])
        got, ok = st.run_chained(samples, sizes)
        assert ok, "the recorded plans outgrew their bounds at density %g" % density
        st.check(got, st.oracle(samples, sizes), batch)
    # full grids (no background rows); should they outgrow the bounds they are planned again the exact way,
    # after which the bounds hold
    for rounds in range(2):
        samples, nSites = draw(5, 1.0)
        st.build(samples, nSites, sizes[0])
        got, ok = st.run_chained(samples, sizes)
        assert ok or rounds == 0
        if not ok:
            got = st.run(samples, sizes)
        st.check(got, st.oracle(samples, sizes), 5)


def test_outgrown_bounds_are_reported_and_raised(scn, ctx):
    rng = np.random.default_rng(5)
    st = Stack(scn, ctx, 2, [("sq", 2, 1, 1), ("sq", 3, 2, 1), ("sq", 2, 1, 1)])
    sizes = st.sizes(19)
    for density, expect in ((0.03, None), (0.035, True), (0.8, False), (0.75, True), (0.02, True)):
        samples, nSites = brute.random_samples(rng, 6, 2, sizes[0], density)
        st.build(samples, nSites, sizes[0])
        if expect is None:
            got = st.run(samples, sizes)
        else:
            got, ok = st.run_chained(samples, sizes)
            assert ok == expect
            if not ok:
                with pytest.raises(scn.ScnError):
                    got[0][0].info()["nSpatialSites"] < 0 or got[0][0].fill(got[1][0], got[1][1], 1)
                got = st.run(samples, sizes)
        st.check(got, st.oracle(samples, sizes), 6)


def test_chained_equals_one_by_one_on_strokes(scn, ctx):
    """The 2-D net's own geometry (five C2 + MP3/2 levels over a 126 field) on stroke-like samples."""
    from conftest import load_scn  # noqa: F401
    from sparseconvnet_archived_amd import synthetic
    cfg = synthetic.config(2, batch=24)
    layers = [("sq", 2, 1, 1), ("sq", 3, 2, 1)] * 5
    st = Stack(scn, ctx, 2, layers)
    sizes = st.sizes(2)
    assert sizes[0] == 126
    for seed in (1, 2, 3):
        samples = synthetic.make_samples(cfg, seed)
        S, K, R, bg, feats, n = synthetic.codify(samples, 2, cfg.lattice, 126, cfg.nInputFeatures)
        per = [(int(bg[i]), {}) for i in range(len(samples))]
        for s, k, r in zip(S, K, R):
            per[int(s)][1][int(k)] = int(r)
        st.build(per, n, 126)
        if seed == 1:
            got = st.run(per, sizes)
        else:
            got, ok = st.run_chained(per, sizes)
            assert ok
        st.check(got, st.oracle(per, sizes), len(per))


def test_a_sample_too_large_for_the_lds_is_planned_layer_by_layer(scn, ctx):
    """A 300 x 300 field holds 90000 sites; a sample with a third of them active does not fit the
    workgroup's arena.  The chain reports it like an outgrown bound."""
    rng = np.random.default_rng(4)
    st = Stack(scn, ctx, 2, [("sq", 2, 1, 1), ("sq", 3, 3, 1)])
    sizes = st.sizes(100)
    assert sizes[0] == 301
    for density, fits in ((0.3, None), (0.28, False), (0.01, True)):
        samples, nSites = brute.random_samples(rng, 3, 2, sizes[0], density)
        st.build(samples, nSites, sizes[0])
        if fits is None:
            got = st.run(samples, sizes)
        else:
            got, ok = st.run_chained(samples, sizes)
            assert ok == fits
            if not ok:
                got = st.run(samples, sizes)
        st.check(got, st.oracle(samples, sizes), 3)


def test_a_layer_that_cannot_join_continues_from_recorded_plans(scn, ctx):
    """Fractional max-pooling regions are not recorded: the plans before them run, and the pooling layer reads
    grids whose table and mask are built from the entry list while their counts are still deferred."""
    rng = np.random.default_rng(9)
    d, sizes = 2, [14, 13, 9]
    src, conv, pool = scn.Grids(ctx), scn.Grids(ctx), scn.Grids(ctx)
    ticksL = np.ascontiguousarray(np.tile(np.array([0, 1, 3, 4, 6, 7, 9, 10, 11], np.int32), (4, d, 1)))
    ticksR = np.ascontiguousarray(ticksL + 2)
    import ctypes as C
    for rec in (False, True, True):
        samples, nSites = brute.random_samples(rng, 4, d, sizes[0], 0.2)
        scn.clear_many(ctx, [src, conv, pool])
        s, k, r, bg = flatten_samples(samples)
        src.build(4, d, sizes[0], s, k, r, bg, nSites)
        og1, o_rules1, o_n1 = orc.rules_square(oracle_grids(samples), d, 14, 13, 2, 1, 1)
        og2, o_rules2, o_n2 = orc.rules_fmp(og1, d, 13, 9, 2, ticksL, ticksR, True)
        if rec:
            scn.defer_counts(ctx, True)
            scn.chain_rules(ctx, True)
        g1, rules1, n1, w1 = scn.rules_square(ctx, src, 14, 13, 2, 1, 1, out=conv)
        # (the binding's plan_fmp asks the input grids for their batch size, which deferred counts forbid)
        n2 = C.c_int64()
        rc = scn.lib().scn_rules_fmp_plan(ctx.h, g1.h, pool.h, 13, 9, 2, ticksL.ctypes.data_as(C.c_void_p),
                                          ticksR.ctypes.data_as(C.c_void_p), C.byref(n2))
        assert rc == scn.OK, scn.lib().scn_last_error()
        w2 = pool.rules_width()
        rules2 = ctx.empty(max(n2.value * w2, 1), np.int32)
        g1.fill(pool, rules2, n2.value * w2)
        g2 = pool
        if rec:
            scn.chain_rules(ctx, False)
            scn.defer_counts(ctx, False)
            assert scn.settle(ctx)
            assert scn.chain_count(ctx)[1] == plans + 1  # the convolution's plan only
        plans = scn.chain_count(ctx)[1]
        assert g1.info()["nSpatialSites"] == o_n1 and g2.info()["nSpatialSites"] == o_n2
        assert np.array_equal(rules1.download()[: o_n1 * w1], o_rules1)
        assert np.array_equal(rules2.download()[: o_n2 * w2], o_rules2)
        assert_same_grids(g1, og1)
        assert_same_grids(g2, og2)


def test_find_on_recorded_grids(scn, ctx):
    samples = [(0, {7: 1, 6: 2, 19: 3}), (4, {0: 5})]
    src, out = scn.Grids(ctx), scn.Grids(ctx)
    for rec in (False, True):
        s, k, r, bg = flatten_samples(samples)
        src.build(2, 2, 5, s, k, r, bg, 6)
        if rec:
            scn.defer_counts(ctx, True)
            scn.chain_rules(ctx, True)
        g, rules, n, w = scn.rules_square(ctx, src, 5, 4, 2, 1, 1, out=out)
        if rec:
            scn.chain_rules(ctx, False)
            scn.defer_counts(ctx, False)
            assert scn.settle(ctx)
        # sample 0: outputs in first-touch order 0,1,4,5 (key 6), 2,6 (key 7), 11,15 (key 19); then its background row
        assert g.find([0, 0, 0, 0, 1, 1], [0, 5, 2, 15, 0, 1]).tolist() == [0, 3, 4, 7, 9, -1]


def test_a_sample_is_shared_out_by_its_own_size_not_the_last_batch_s(scn):
    """How many workgroups a sample is worth is planned from the sites a sample of the batch before had at each level:
    one small drawing after a batch of forty is shared out as after a single one."""
    layers = [("sq", 2, 1, 1), ("sq", 3, 2, 1)] * 5
    sample = {126 * (40 + i % 5) + 40 + i: i + 1 for i in range(24)}
    splits = []
    for before in (1, 40):
        ctx = scn.Context()
        st = Stack(scn, ctx, 2, layers)
        sizes = st.sizes(2)
        many = [(25 * b, {k: r + 25 * b for k, r in sample.items()}) for b in range(before)]
        st.build(many, 25 * before, sizes[0])
        st.run(many, sizes)
        one = [(0, dict(sample))]
        st.build(one, 25, sizes[0])
        got, ok = st.run_chained(one, sizes)
        assert ok
        st.check(got, st.oracle(one, sizes), 1)
        splits.append(scn.chain_split(ctx))
    assert splits[0] == splits[1] and 1 <= splits[0][0] < 24, splits


@pytest.mark.parametrize("d,layers,batch,parts,slabs", [
    (3, [("sq", 2, 1, 1), ("sq", 2, 2, 1)] * 4, 5, (12, 24), (14, 48)),  # 47^3: layers in slabs, levels in slabs
    (2, [("sq", 2, 1, 1), ("sq", 3, 2, 1)] * 5, 3, (4, 24), (11, 11)),   # 126 x 126, ten layers: a wavefront a level
    (2, [("sq", 2, 1, 1), ("sq", 3, 2, 1)] * 5, 100, (1, 1), (11, 11)),  # enough samples: a workgroup each
    (1, [("sq", 3, 1, 1), ("sq", 2, 2, 1)], 4, (1, 24), (0, 0))])        # one dimension: level after level
def test_samples_are_shared_out_and_stay_the_same(scn, d, layers, batch, parts, slabs):
    ctx = scn.Context()
    st = Stack(scn, ctx, d, layers)
    sizes = st.sizes(2)
    n, rng, samples, row = sizes[0], np.random.default_rng(d + batch), [], 0
    for b in range(batch):  # thick shells and strokes, in rows of no order; samples unlike in size
        at = np.stack(np.meshgrid(*[np.arange(n)] * d, indexing="ij"), -1).reshape(-1, d)
        off = np.abs(np.linalg.norm(at - rng.uniform(0.4, 0.6, d) * n, axis=1) - rng.uniform(0.15, 0.25) * n)
        keys = rng.permutation(np.flatnonzero(off < 0.5 + 0.1 * (b % 3)))
        samples.append((row, {int(k): row + 1 + i for i, k in enumerate(keys)}))
        row += len(keys) + 1
    st.build(samples, row, n)
    st.run(samples, sizes)
    for _ in range(2):  # the second time with LDS for what was seen
        st.build(samples, row, n)
        got, ok = st.run_chained(samples, sizes)
        assert ok
        split = scn.chain_split(ctx)
        print("split", split, flush=True)
        assert parts[0] <= split[0] <= parts[1] and slabs[0] <= split[1] <= slabs[1], split
        st.check(got, st.oracle(samples, sizes), batch)
