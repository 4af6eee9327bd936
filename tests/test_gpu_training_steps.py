"""The pieces a training batch is put together from: the activation's derivative over the outputs of the pooling behind
the layer (scn_activation_backward_to) against the derivative over the layer's own rows, and the momentum step of many
tensors in one launch against the formula in float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["RELU", "LEAKYRELU", "PRELU", "TANH", "NOSIGMOID"])
@pytest.mark.parametrize("rows,outs,ps,N", [(1, 1, 1, 1), (40, 17, 4, 3), (900, 400, 9, 32), (5000, 1300, 8, 100),
                                            (70000, 30001, 9, 64)])
def test_derivative_over_the_outputs_of_a_pooling(scn, ctx, act, rows, outs, ps, N):
    print("activation ahead", act, rows, outs, ps, N, flush=True)
    rng = np.random.default_rng(rows + N)
    a = getattr(scn, act, 0)
    y = rng.standard_normal((rows, N)).astype(np.float32)
    if act == "TANH":
        y = np.tanh(y)
    if act == "RELU":
        y = np.maximum(y, 0)
    pr = rng.uniform(0.1, 0.4, N).astype(np.float32)
    rules = rng.integers(0, rows, (outs, ps)).astype(np.int32)
    dp = rng.standard_normal((outs, N)).astype(np.float32)
    d_y, d_rules, d_pr, d_dp = (ctx.array(v) for v in (y, rules, pr, dp))
    pooled, choice = ctx.empty((outs, N), np.float32), ctx.empty((outs, N), np.int32)
    ctx.maxpool(d_y, pooled, d_rules, outs, ps, N, choice)
    got = []
    for ahead in (False, True):
        dy = ctx.array(np.zeros((rows, N), np.float32))
        db, dpr = ctx.array(np.full(N, 5, np.float32)), ctx.array(np.full(N, 5, np.float32))
        prelu = (d_pr, dpr) if act == "PRELU" else (None, None)
        if ahead:
            spread = ctx.empty((outs, N), np.float32)
            ctx.activation_backward_to(pooled, d_dp, spread, outs, N, a, prelu[0], db, prelu[1])
            assert np.array_equal(d_dp.download(), dp)  # left as it is
            ctx.maxpool_backward(dy, spread, outs, N, choice)
        else:
            ctx.maxpool_backward(dy, d_dp, outs, N, choice)
            ctx.activation_backward(d_y, dy, rows, N, a, prelu[0], db, prelu[1])
        got.append((dy.download(), db.download(), dpr.download()))
    # (up to `outs` numbers of order one are added in another order: half an ulp of the partial sum each)
    for u, v in zip(*got):
        bound = 2.0 ** -23 * np.sqrt(outs) * 8 * max(1.0, np.abs(u).max())
        assert np.abs(u - v).max() <= bound, (np.abs(u - v).max(), bound)
    assert np.abs(got[0][1]).max() > 0


@pytest.mark.parametrize("count", [1, 5, 48])
def test_momentum_step_of_many_tensors(scn, ctx, count):
    rng = np.random.default_rng(count)
    sizes = [int(n) for n in rng.choice([1, 255, 256, 257, 5000], count)]
    host = [[rng.standard_normal(n).astype(np.float32) for _ in range(3)] for n in sizes]
    dev = [[ctx.array(a) for a in t] for t in host]
    ctx.nag_update_many([(d, m, w, n, i % 2) for i, ((d, m, w), n) in enumerate(zip(dev, sizes))], 0.01, 0.9, True)
    for i, ((d, m, w), (dd, dm, dw)) in enumerate(zip(host, dev)):
        d, m, w = (a.astype(np.float64) for a in (d, m, w))
        m2 = 0.9 * m - 0.01 * (1 - 0.9) * d
        w2 = w - m * 0.9 + m2 * (1 + 0.9)
        if i % 2:
            w2 = np.maximum(w2, 0.001)
        assert np.abs(dm.download() - m2).max() <= 4 * 2.0 ** -24 * 4 and np.abs(dw.download() - w2).max() <= 8 * 2.0 ** -24 * 8
        assert not dd.download().any()
