"""Grids built from sites whose neighbours share words of the mask, at the edges of the runs that make one atomic, and
the copy of a batch's features in the same launch."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

#  samples, field, how the sites come, sites of a sample (none: an empty sample list)
FORMS = [(1, 3, "sorted", 5), (2, 63, "runs", 300), (3, 64, "runs", 257), (2, 95, "reversed", 2000), (5, 40, "shuffled", 1600),
         (1, 16, "full", 256), (1200, 129, "runs", 40), (2, 9, "none", 0), (0, 9, "none", 0)]


@pytest.mark.parametrize("batch,n,order,per", FORMS)
@pytest.mark.parametrize("bytes_,at,to", [(0, 0, 0), (4, 0, 0), (1000, 0, 0), (1004, 4, 0), (1008, 8, 8), (70004, 0, 0), (33, 1, 3)])
def test_sites_and_copy(scn, ctx, batch, n, order, per, bytes_, at, to):
    print("grid build", batch, n, order, per, bytes_, flush=True)
    rng = np.random.default_rng(n + per)
    keys = []
    for b in range(batch):
        if order == "runs":  # pieces of rows, of 1 to 40 sites
            k = np.unique(np.concatenate([s + np.arange(rng.integers(1, 41)) for s in rng.integers(0, n * n - 40, per)]))[:per]
        else:
            k = np.sort(rng.choice(n * n, per, replace=False))
        k = k[::-1] if order == "reversed" else rng.permutation(k) if order == "shuffled" else k
        keys.append(k)
    key = np.concatenate(keys + [np.zeros(0, np.int64)]).astype(np.int64)
    sample = np.repeat(np.arange(batch), [len(k) for k in keys]).astype(np.int32)
    row = (np.arange(len(key)) + 1).astype(np.int32)
    bg = rng.integers(0, 9, batch).astype(np.int32)
    src = rng.integers(0, 256, bytes_ + at + 64).astype(np.uint8)
    dst = np.zeros(bytes_ + to + 64, np.uint8)
    d_src, d_dst = ctx.array(src, np.uint8), ctx.array(dst, np.uint8)
    arrays = [ctx.array(a if len(a) else np.zeros(1, t), t)
              for a, t in ((sample, np.int32), (key, np.int64), (row, np.int32), (bg, np.int32))]
    g, out = scn.Grids(ctx), scn.Grids(ctx)
    scn._check(scn.lib().scn_grids_build_copy(ctx.h, g.h, batch, 2, n, *[a.ptr for a in arrays[:3]], len(key), arrays[3].ptr,
                                              len(key) + 1, C.c_void_p(d_dst.ptr + to), C.c_void_p(d_src.ptr + at), bytes_))
    dst[to:to + bytes_] = src[at:at + bytes_]
    assert np.array_equal(d_dst.download(), dst)
    s, k, r, gotBg = g.download()
    want = np.lexsort((key, sample))
    got = np.lexsort((k, s))
    assert np.array_equal(s[got], sample[want]) and np.array_equal(k[got], key[want]) and np.array_equal(r[got], row[want])
    assert np.array_equal(gotBg, bg)
    if len(key):
        assert np.array_equal(g.find(sample, key), row)
        # the mask, through a pooling of windows of one site: a row for each site, and one for
        # the background of each sample that has any
        assert g.plan_square(out, n, n, 1, 1, 1) == len(key) + sum(len(k) < n * n for k in keys)
