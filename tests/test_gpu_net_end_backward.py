"""A net's end in a training batch: the classifier with its cost's gradient in one launch (the bits of the three calls), and
backwards the classifier's input gradient, spread over the pooled rows with the activation's derivative, in another."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (samples, channels, classes, rows of a sample at most): odd numbers of samples, channels that are no whole round of the
# workgroup's rows of W, most channels and classes, more rows than are taken at a time
SHAPES = [(1, 4, 4, 1), (33, 128, 40, 8), (100, 192, 100, 4), (7, 36, 12, 9), (61, 800, 100, 9), (2, 1024, 128, 20), (513, 20, 128, 16)]


def pooled_rows(rng, M, S):
    """rules of M samples (some without a row) that name every row once, and how many rows there are (two more than named)"""
    count = rng.integers(0, S + 1, M)
    count[0] = S
    order = rng.permutation(count.sum() + 2).astype(np.int32)
    rules, at = np.full((M, S), -1, np.int32), 0
    for b in range(M):
        rules[b, :count[b]] = order[at:at + count[b]]
        at += count[b]
    return rules, len(order), count


@pytest.mark.parametrize("M,K,N,S", [s for s in SHAPES if s[0] <= 512])
def test_classifier_and_gradient(scn, ctx, M, K, N, S):
    if not scn.lib().scn_terminal_classifier_supported(M, K, N):
        pytest.skip("not one for this kernel")
    rng = np.random.default_rng(M + K)
    rules, rows, count = pooled_rows(rng, M, S)
    rules[count == 0, 0] = 0  # (a sample pools something)
    d_x, d_rules = ctx.array(rng.standard_normal((rows, K), dtype=np.float32)), ctx.array(rules)
    d_W, d_B = ctx.array((rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)), ctx.array(rng.standard_normal(N, dtype=np.float32))
    d_labels = ctx.array(rng.integers(0, N, M).astype(np.int32))
    outs = [[ctx.array(np.full((M + 3, w), 7, np.float32)) for w in (K, N, N, N)] for _ in range(2)]
    pooled, probs, copy, delta = outs[0]
    ctx.terminal_classifier_train(d_x, d_rules, M, S, pooled, d_W, d_B, probs, copy, K, N, d_labels, delta)
    pooled, probs, copy, delta = outs[1]
    ctx.terminal_classifier(d_x, d_rules, M, S, pooled, d_W, d_B, probs, copy, K, N)
    scn.lib().scn_softmax_grad(ctx.h, probs.ptr, d_labels.ptr, delta.ptr, M, N)
    for a, b in zip(*outs):
        a, b = a.download(), b.download()
        assert np.array_equal(a, b) and np.all(a[M:] == 7)


@pytest.mark.parametrize("M,K,N,S", SHAPES)
@pytest.mark.parametrize("act", ["NOSIGMOID", "RELU", "VLEAKYRELU", "LEAKYRELU", "PRELU", "TANH", "SIGMOID"])
def test_terminal_gradient(scn, ctx, M, K, N, S, act):
    rng = np.random.default_rng(M + N)
    a = getattr(scn, act)
    rules, rows, _ = pooled_rows(rng, M, S)
    delta, W = rng.standard_normal((M, N), dtype=np.float32), rng.standard_normal((K, N), dtype=np.float32)
    y = rng.standard_normal((rows, K), dtype=np.float32)
    if act in ("TANH", "SIGMOID"):
        y = np.tanh(y) if act == "TANH" else 1 / (1 + np.exp(-y))
    slopes, start = rng.uniform(0.1, 0.4, K).astype(np.float32), rng.standard_normal(K, dtype=np.float32)
    d_delta, d_W, d_rules, d_y, d_slopes = (ctx.array(x) for x in (delta, W, rules, y, slopes))
    din, dpooled, dprelu = ctx.array(np.zeros((rows, K), np.float32)), ctx.array(np.full((M + 2, K), 7, np.float32)), ctx.array(start)
    prelu = act == "PRELU"
    ctx.terminal_gradient(d_delta, d_W, dpooled, d_rules, M, S, din, d_y, a, d_slopes if prelu else None, dprelu if prelu else None, K, N)
    want = delta.astype(np.float64) @ W.T.astype(np.float64)
    scale = np.abs(delta).astype(np.float64) @ np.abs(W).T.astype(np.float64)
    got = dpooled.download()
    assert np.all(got[M:] == 7) and np.all(np.abs(got[:M] - want) <= N * 2.0 ** -24 * scale)
    # spread and derivative of what the kernel has as the pooled gradient, against the calls that do it one by one
    two, db, dtwo = ctx.array(np.zeros((rows, K), np.float32)), ctx.array(np.zeros(K, np.float32)), ctx.array(np.zeros(K, np.float32))
    ctx.terminal_pool_backward(two, dpooled, d_rules, M, K, S)
    spread = two.download()
    assert scn.lib().scn_activation_backward(ctx.h, d_y.ptr, two.ptr, rows, K, a, d_slopes.ptr, db.ptr, dtwo.ptr) == 0
    assert np.array_equal(din.download(), two.download())
    if prelu:
        terms = np.where(y > 0, 0, spread.astype(np.float64) * y / slopes)
        assert np.all(np.abs(dprelu.download() - start - terms.sum(0)) <= 2.0 ** -21 * (np.abs(terms).sum(0) + np.abs(start)))
    else:
        assert np.array_equal(dprelu.download(), start)


# what the backward pass begins with beside the classifier: odd numbers of 256-lane blocks, buffers off 16 bytes, none, filters alone
@pytest.mark.parametrize("M,K,N,S", [(1, 4, 4, 1), (33, 128, 40, 8), (100, 192, 100, 4)])
@pytest.mark.parametrize("sizes,filters", [([], [(1, 3, 33)]), ([1025, 0, 3], []), ([70000], [(4, 31, 5), (8, 96, 32), (4, 32, 64)])])
def test_classifier_with_the_beginning(scn, ctx, M, K, N, S, sizes, filters):
    rng = np.random.default_rng(M + K)
    rules, rows, count = pooled_rows(rng, M, S)
    rules[count == 0, 0] = 0
    d_x, d_rules = ctx.array(rng.standard_normal((rows, K), dtype=np.float32)), ctx.array(rules)
    d_W, d_B = ctx.array((rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)), ctx.array(rng.standard_normal(N, dtype=np.float32))
    d_labels = ctx.array(rng.integers(0, N, M).astype(np.int32))
    outs = [[ctx.array(np.full((M + 3, w), 7, np.float32)) for w in (K, N, N, N)] for _ in range(2)]
    bufs = [ctx.array(np.full(n + 4, 7, np.int32)) for n in sizes]
    Ws = [rng.standard_normal(f, dtype=np.float32) for f in filters]
    turned, held = [ctx.array(np.full(W.size + 4, 7, np.float32)) for W in Ws], [ctx.array(W) for W in Ws]
    ptrs = (C.c_void_p * max(1, len(sizes)))(*[b.ptr for b in bufs])
    words = (C.c_size_t * max(1, len(sizes)))(*sizes)
    items = (scn.FilterItem * max(1, len(filters)))(*[scn.FilterItem(w.ptr, o.ptr, *f) for w, o, f in zip(held, turned, filters)])
    print("classifier and beginning", M, K, N, S, sizes, filters, flush=True)
    pooled, probs, copy, delta = outs[0]
    scn._check(scn.lib().scn_terminal_classifier_begin(ctx.h, d_x.ptr, d_rules.ptr, M, S, pooled.ptr, d_W.ptr, d_B.ptr, probs.ptr, copy.ptr,
                                                       K, N, 1.0, d_labels.ptr, delta.ptr, ptrs, words, len(sizes), items, len(filters)))
    pooled, probs, copy, delta = outs[1]
    ctx.terminal_classifier_train(d_x, d_rules, M, S, pooled, d_W, d_B, probs, copy, K, N, d_labels, delta)
    for a, b in zip(*outs):
        assert np.array_equal(a.download(), b.download())
    for b, n in zip(bufs, sizes):
        assert np.all(b.download()[:n] == 0) and np.all(b.download()[n:] == 7)
    for W, o in zip(Ws, turned):
        got = o.download()
        assert np.array_equal(got[:-4].reshape(W.shape[0], W.shape[2], W.shape[1]), W.transpose(0, 2, 1)) and np.all(got[-4:] == 7)


def test_what_is_not_supported_is_refused(scn, ctx):
    L = scn.lib()
    for K, N in ((1028, 100), (128, 132), (6, 100), (128, 10)):
        assert not L.scn_terminal_gradient_supported(K, N)
        assert L.scn_terminal_gradient(ctx.h, None, None, None, None, 1, 1, None, None, scn.RELU, None, None, K, N) != 0
