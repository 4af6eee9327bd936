"""Grids emptied by scn_grids_clear_many take the mask that the build before has emptied: nothing of a batch is left in the
next or the one after it, and a captured graph keeps the mask it was captured with."""
import numpy as np
import pytest

import brute
import oracle as orc
from gpu_util import assert_same_grids, flatten_samples, oracle_grids
from test_gpu_capture import Graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,side", [(2, 34), (3, 14)])
def test_batch_after_batch(scn, ctx, d, side):
    """more sites and fewer, none at all, a mask outgrown and one too large for a spare"""
    rng = np.random.default_rng(side)
    grids, out = scn.Grids(ctx), scn.Grids(ctx)
    huge = 3300 if d == 2 else 230  # (batch 1: more than 1 MB of mask)
    for batch, n, density in [(5, side, 0.2), (5, side, 0.01), (4, side, 0.3), (0, side, 0.1), (5, side, 0.02), (30, side, 0.1),
                              (30, side, 0.01), (1, huge, 2e-4 if d == 2 else 1e-4), (6, side, 0.1), (6, side, 0.02)]:
        samples, nSites = brute.random_samples(rng, batch, d, n, density)
        s, k, r, bg = flatten_samples(samples)
        scn.clear_many(ctx, [grids, out])
        print("batch", batch, n, len(k), flush=True)
        grids.build(batch, d, n, s, k, r, bg, nSites)
        og = oracle_grids(samples)
        assert_same_grids(grids, og)
        o_out, o_rules, o_n = orc.rules_square(og, d, n, n - 1, 2, 1, 1)
        d_out, d_rules, rows, w = scn.rules_square(ctx, grids, n, n - 1, 2, 1, 1, out=out)
        assert rows == o_n and np.array_equal(d_rules.download()[:rows * w], o_rules)
        assert_same_grids(d_out, o_out)


def test_a_graph_keeps_its_mask(scn, ctx):
    rng = np.random.default_rng(5)
    L, B, n = scn.lib(), 4, 40
    grids = scn.Grids(ctx)

    def sites(density):
        samples, nSites = brute.random_samples(rng, B, 2, n, density)
        s, k, r, bg = flatten_samples(samples)
        want = np.full((B, n * n), -1, np.int32)
        want[s, k] = r
        return [ctx.array(np.asarray(a, t)) for a, t in zip((s, k, r, bg), (np.int32, np.int64, np.int32, np.int32))], len(k), nSites, want

    everywhere = [ctx.array(np.repeat(np.arange(B, dtype=np.int32), n * n)), ctx.array(np.tile(np.arange(n * n, dtype=np.int64), B))]
    found = ctx.array(np.zeros(B * n * n, np.int32))

    def go(batch):
        arrays, m, nSites, _ = batch
        scn.clear_many(ctx, [grids])
        grids.build_device(B, 2, n, *arrays, m, nSites)
        assert L.scn_grids_find(ctx.h, grids.h, everywhere[0].ptr, everywhere[1].ptr, B * n * n, found.ptr) == 0

    first, second, third = sites(0.3), sites(0.2), sites(0.25)
    for batch in (first, second, first):
        go(batch)
        assert np.array_equal(found.download().reshape(B, -1), batch[3])
    with Graph(ctx) as g:
        go(second)
    for batch in (third, first, third):
        for _ in range(2):
            g.replay(ctx)
            assert np.array_equal(found.download().reshape(B, -1), second[3])
        go(batch)
        assert np.array_equal(found.download().reshape(B, -1), batch[3])
    g.close()
