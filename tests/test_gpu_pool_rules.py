"""Max-pooling whose rules come through LDS, against numpy: whole and part workgroups, rows that two of them share (channels
that do not divide 1024), windows of the sizes compiled in and others, rules that do not fit, scalar channels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,ps,C", [(1, 9, 32), (257, 9, 4), (64, 9, 1024), (33, 9, 1500), (1000, 8, 96), (77, 4, 20), (300, 1, 8),
                                       (41, 27, 64), (300, 27, 4), (5, 32, 2048), (129, 9, 3), (0, 9, 32)])
def test_maxpool(scn, ctx, rows, ps, C):
    rng = np.random.default_rng(rows + ps + C)
    n = 50
    x = np.round(rng.standard_normal((n, C)) * 4).astype(np.float32)  # (ties: the first of them wins)
    rules = rng.integers(-1, n, (rows, ps)).astype(np.int32)
    if rows > 1:
        rules[1] = -1
    y, ch = ctx.empty((max(rows, 1), C), np.float32), ctx.empty((max(rows, 1), C), np.int32)
    print("maxpool", rows, ps, C, flush=True)
    ctx.maxpool(ctx.array(x), y, ctx.array(rules if rows else np.zeros((1, ps), np.int32)), rows, ps, C, ch)
    want, arg = np.zeros((rows, C), np.float32), np.zeros((rows, C), np.int64)
    for r in range(rows):
        named = rules[r][rules[r] >= 0]
        if len(named):
            k = x[named].argmax(0)
            want[r], arg[r] = x[named[k], np.arange(C)], named[k].astype(np.int64) * C + np.arange(C)
    assert np.array_equal(y.download()[:rows], want) and np.array_equal(ch.download()[:rows], arg)
