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
