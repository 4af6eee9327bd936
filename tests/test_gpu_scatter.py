"""Scatter-add through a rule book: every tile, ragged last tiles, channels divided among workgroups, background rows
of many entries (one and more to a tile than are summed in LDS), channels beyond what LDS holds."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


# (entries, channels, background rows)
@pytest.mark.parametrize("count,nIn,backgrounds", [(1, 1, 1), (63, 3, 1), (65, 33, 7), (1000, 513, 6), (129, 1100, 1),
                                                   (32768, 96, 2), (32769, 40, 9), (50001, 160, 3), (60000, 513, 1),
                                                   (327679, 32, 20), (327681, 33, 1), (400003, 5, 12)])
def test_scatter_add(scn, ctx, count, nIn, backgrounds):
    rng = np.random.default_rng(count + nIn)
    rowsIn = max(count // 4, 1) + backgrounds
    # neighbouring entries share rows, as neighbouring windows do
    rules = (np.arange(count) // 4 + rng.integers(0, 8, count)) % rowsIn
    hidden = rng.random(count) < 0.4
    rules[hidden] = rng.integers(0, backgrounds, int(hidden.sum()))
    rules[rng.random(count) < 0.01] = -1
    rules = rules.astype(np.int32)
    print("scatter", count, nIn, flush=True)
    dconv = rng.integers(-3, 4, (count, nIn)).astype(np.float32)  # integers: exact in any order
    before = rng.integers(-3, 4, (rowsIn, nIn)).astype(np.float32)
    d_din = ctx.array(before)
    ctx.gather_rows_backward(d_din, ctx.array(dconv), ctx.array(rules), count, nIn)
    assert np.array_equal(d_din.download(), before + orc.gather_rows_backward(dconv, rules, rowsIn, nIn))


# one entry; channels below, at and past a slice; every tile; windows that share rows, and entries all over the input:
# more rows than a tile has room for
@pytest.mark.parametrize("count,C", [(1, 1), (7, 3), (1000, 31), (16, 32), (65, 33), (9001, 96), (129, 513), (20001, 64),
                                     (70001, 128), (2100001, 1)])
@pytest.mark.parametrize("spread", [False, True])
def test_pooling_gradient(scn, ctx, count, C, spread):
    rng = np.random.default_rng(count + C)
    rowsIn = 2 * count + 9
    row = rng.integers(0, rowsIn, (count, C)) if spread else (2 * np.arange(count)[:, None] + rng.integers(0, 9, (count, C)))
    hidden = rng.random((count, C)) < 0.2
    row[hidden] = (np.broadcast_to(np.arange(count)[:, None] // 300, (count, C)))[hidden]
    choice = (row * C + np.arange(C)).astype(np.int32)
    choice[rng.random((count, C)) < 0.01] = -1
    print("pooling gradient", count, C, spread, flush=True)
    dout = rng.integers(-3, 4, (count, C)).astype(np.float32)  # integers: exact in any order
    before = rng.integers(-3, 4, (rowsIn, C)).astype(np.float32)
    d_din = ctx.array(before)
    ctx.maxpool_backward(d_din, ctx.array(dout), count, C, ctx.array(choice))
    want = before.astype(np.float64).reshape(-1)
    np.add.at(want, choice[choice >= 0], dout[choice >= 0])
    assert np.array_equal(d_din.download().reshape(-1), want)
