"""Weight gradients in two by two tiles through rules: layers of one launch whose columns are whole tiles, half ones and both,
and single ones large enough for them, against 64-bit sums."""
import numpy as np
import pytest
from test_gpu_conv_backward import layer

pytestmark = pytest.mark.gpu


def item(scn, ctx, rng, d, field, window, batch, density, nIn, N):
    g, n, rows, fs, d_rules, bg = layer(scn, ctx, d, field, window, batch, density, field + N)
    positions = ctx.empty((fs, (rows + 15) // 16 * 16), np.int32)
    ctx.rules_inverse_many([(g, d_rules, None, None, positions, rows, n, fs)])
    rules = d_rules.download()
    x, D = rng.standard_normal((n, nIn), dtype=np.float32), rng.standard_normal((rows, N), dtype=np.float32)
    A = np.where(rules[:, :, None] >= 0, x[np.maximum(rules, 0)], 0).reshape(rows, fs * nIn)
    return (ctx.array(x), positions, fs, nIn, ctx.array(D), rows, N), A, D


def compare(A, D, dW, db, start):
    """sums of sixteen million products at most, in parts of sixteen rows by planes: as test_gpu_conv_backward"""
    A, D = A.astype(np.float64), D.astype(np.float64)
    assert np.all(np.abs(dW.download() - start[:-1] - A.T @ D) <= 2e-6 * (np.abs(A).T @ np.abs(D) + np.abs(start[:-1])))
    assert np.all(np.abs(db.download() - start[-1] - D.sum(0)) <= 2e-6 * (np.abs(D).sum(0) + np.abs(start[-1])))


# columns: one tile's worth and less, half a tile and no more behind whole ones; rows: fewer than a wavefront's, some
# wavefronts', several ranges'; dW's rows: half a tile, no whole tile
@pytest.mark.parametrize("first,second", [((1, 9, 2, 1, 0.3, 16, 96), (2, 12, 2, 2, 0.2, 32, 36)),
                                          ((2, 40, 2, 20, 0.15, 32, 68), (2, 40, 2, 9, 0.15, 3, 32)),
                                          ((3, 12, 3, 4, 0.1, 20, 128), (2, 30, 3, 6, 0.3, 64, 100)),
                                          ((2, 60, 2, 30, 0.2, 96, 160), (2, 9, 2, 1, 0.3, 64, 32))])
def test_several_layers(scn, ctx, first, second):
    rng = np.random.default_rng(first[-1])
    made = [item(scn, ctx, rng, *first), item(scn, ctx, rng, *second)]
    print("weight gradients of", [(i[2], i[3], i[5], i[6]) for i, _, _ in made], flush=True)
    starts = [rng.standard_normal((A.shape[1] + 1, D.shape[1]), dtype=np.float32) for _, A, D in made]
    out = [(ctx.array(s[:-1]), ctx.array(s[-1])) for s in starts]
    ctx.AtB_many([(x, p, fs, nIn, D, dW, db, M, N) for ((x, p, fs, nIn, D, M, N), _, _), (dW, db) in zip(made, out)])
    for (_, A, D), s, (dW, db) in zip(made, starts, out):
        compare(A, D, dW, db, s)


@pytest.mark.parametrize("shape", [(3, 22, 3, 4, 0.02, 32, 128), (2, 90, 3, 14, 0.1, 128, 96)])
def test_one_layer(scn, ctx, shape):
    rng = np.random.default_rng(shape[-1])
    (x, p, fs, nIn, d_D, M, N), A, D = item(scn, ctx, rng, *shape)
    print("weight gradient of", fs, nIn, M, N, flush=True)
    start = rng.standard_normal((fs * nIn + 1, N), dtype=np.float32)
    dW, db = ctx.array(start[:-1]), ctx.array(start[-1])
    ctx.AtB_many([(x, p, fs, nIn, d_D, dW, db, M, N)])
    compare(A, D, dW, db, start)
