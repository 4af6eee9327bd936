"""Memory that is written whole without being cleared first: fills at any alignment, the masks and scan states of rule
books whose objects were used for other sites before."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 5, 1023, 4097, 300001])
@pytest.mark.parametrize("off", [0, 1, 2, 3])
def test_fill_touches_its_words_only(scn, ctx, n, off):
    d = ctx.array(np.arange(n + 8, dtype=np.int32))
    print("fill", n, off, flush=True)
    assert scn.lib().scn_fill32(ctx.h, d.ptr + 4 * off, 0x12345678, n) == 0
    want = np.arange(n + 8, dtype=np.int32)
    want[off:off + n] = 0x12345678
    assert np.array_equal(d.download(), want)


@pytest.mark.parametrize("sizes", [(1,), (0, 5, 0), (1023, 1, 70001, 0, 4096, 3) * 5])
def test_fill_of_several_buffers(scn, ctx, sizes):
    import ctypes
    bufs = [ctx.array(np.arange(n + 5, dtype=np.int32)) for n in sizes]
    print("fills", sizes, flush=True)
    ptrs = (ctypes.c_void_p * len(sizes))(*[b.ptr + 4 * (i % 4) for i, b in enumerate(bufs)])
    assert scn.lib().scn_fill32_many(ctx.h, ptrs, (ctypes.c_size_t * len(sizes))(*sizes), len(sizes), 7) == 0
    for i, (b, n) in enumerate(zip(bufs, sizes)):
        want = np.arange(n + 5, dtype=np.int32)
        want[i % 4:i % 4 + n] = 7
        assert np.array_equal(b.download(), want), i


# more entries than one workgroup scans, with and without tiled windows, and few; a denser set of sites before
@pytest.mark.parametrize("d,field,samples,size,stride", [(3, 40, 9, 3, 1), (3, 40, 9, 2, 2), (2, 121, 33, 3, 2), (2, 20, 3, 2, 1)])
def test_rule_books_on_used_objects(scn, ctx, d, field, samples, size, stride):
    out = (field - size) // stride + 1
    field = (out - 1) * stride + size
    rng = np.random.default_rng(field + size)
    used, results = [scn.Grids(ctx), scn.Grids(ctx)], []
    for share in (0.4, 0.15):
        active = rng.random((samples, field ** d)) < share
        sample, key = (a.astype(t) for a, t in zip(np.nonzero(active), (np.int32, np.int64)))
        per = active.sum(1)
        row = (np.arange(len(key)) + sample + 1).astype(np.int32)
        bg = (np.concatenate([[0], np.cumsum(per)[:-1]]) + np.arange(samples)).astype(np.int32)
        n = len(key) + samples
        results = []
        for gin, gout in (used, (scn.Grids(ctx), scn.Grids(ctx))):
            gin.build_device(samples, d, field, *(ctx.array(a) for a in (sample, key, row, bg)), len(key), n)
            rows = gin.plan_square(gout, field, out, size, stride)
            rules = ctx.empty((rows * size ** d,), np.int32)
            gin.fill(gout, rules, rows * size ** d)
            gnext = scn.Grids(ctx)  # what stands on the mask of the output
            rows2 = gout.plan_square(gnext, out, out - 1, 2, 1)
            rules2 = ctx.empty((rows2 * 2 ** d,), np.int32)
            gout.fill(gnext, rules2, rows2 * 2 ** d)
            results.append((rows, rules.download(), rows2, rules2.download()))
        mask = active.reshape((samples,) + (field,) * d)
        for axis in range(1, d + 1):
            mask = np.logical_or.reduce([np.take(mask, np.arange(out) * stride + o, axis) for o in range(size)])
        full = (mask.reshape(samples, -1).sum(1) == out ** d).sum()
        assert results[0][0] == mask.sum() + samples - full or results[0][0] == mask.sum() + samples
        assert all(np.array_equal(a, b) for a, b in zip(*results))


# buffers and filters in one launch, either without the other; buffers that end off 16 bytes, none, one past a workgroup's share
@pytest.mark.parametrize("sizes", [[], [1], [1025, 0, 70000, 3]])
@pytest.mark.parametrize("filters", [[], [(4, 32, 64)], [(1, 3, 33), (8, 96, 32), (4, 31, 5)]])
def test_a_backward_pass_begins(scn, ctx, sizes, filters):
    rng = np.random.default_rng(len(sizes) + 8 * len(filters))
    bufs = [ctx.array(np.full(n + 4, 7, np.int32)) for n in sizes]
    Ws = [rng.standard_normal((fs, nIn, N), dtype=np.float32) for fs, nIn, N in filters]
    outs = [ctx.array(np.full(W.size, 7, np.float32)) for W in Ws]
    held = [ctx.array(W) for W in Ws]
    ptrs = (C.c_void_p * max(1, len(sizes)))(*[b.ptr for b in bufs])
    words = (C.c_size_t * max(1, len(sizes)))(*sizes)
    items = (scn.FilterItem * max(1, len(filters)))(*[scn.FilterItem(w.ptr, o.ptr, *f) for w, o, f in zip(held, outs, filters)])
    print("backward begins", sizes, filters, flush=True)
    scn._check(scn.lib().scn_gradients_begin(ctx.h, ptrs, words, len(sizes), items, len(filters)))
    for b, n in zip(bufs, sizes):
        got = b.download()
        assert np.all(got[:n] == 0) and np.all(got[n:] == 7)
    for W, o in zip(Ws, outs):
        assert np.array_equal(o.download().reshape(W.shape[0], W.shape[2], W.shape[1]), W.transpose(0, 2, 1))


@pytest.mark.parametrize("batch,N", [(1, 3), (100, 100), (257, 40)])
def test_classifier_gradient_with_a_copy(scn, ctx, batch, N):
    rng = np.random.default_rng(batch)
    p, labels = rng.random((batch, N), dtype=np.float32), rng.integers(0, N, batch).astype(np.int32)
    delta, copy = (ctx.array(np.full((batch, N), 7, np.float32)) for _ in range(2))
    held = ctx.array(p), ctx.array(labels)
    print("gradient and copy", batch, N, flush=True)
    scn._check(scn.lib().scn_softmax_grad_copy(ctx.h, held[0].ptr, held[1].ptr, delta.ptr, batch, N, copy.ptr))
    want = p.copy()
    want[np.arange(batch), labels] -= 1
    assert np.array_equal(delta.download(), want) and np.array_equal(copy.download(), p)
