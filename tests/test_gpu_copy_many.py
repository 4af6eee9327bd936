"""scn_copy_many: the bytes of several copies, of any size and alignment, and nothing beside them."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,skew", [([], 0), ([0, 5], 0), ([1, 16, 17, 4096 * 16 * 3 + 5], 0), ([40000, 33, 0, 3000000], 4),
                                        ([7, 64, 100, 129, 1, 15, 2048, 5000], 1)])
def test_copies(scn, ctx, sizes, skew):
    rng = np.random.default_rng(len(sizes))
    src = [ctx.array(rng.integers(0, 256, n + 32).astype(np.uint8)) for n in sizes]
    dst = [ctx.array(np.full(n + 32, 9, np.uint8)) for n in sizes]
    n = len(sizes)
    to, frm = (C.c_void_p * max(n, 1))(*[d.ptr + skew for d in dst]), (C.c_void_p * max(n, 1))(*[s.ptr + (skew & 1) for s in src])
    assert scn.lib().scn_copy_many(ctx.h, to, frm, (C.c_size_t * max(n, 1))(*sizes), n) == 0
    for s, d, k in zip(src, dst, sizes):
        got, from_ = d.download(), s.download()[skew & 1:]
        assert np.array_equal(got[skew:skew + k], from_[:k]) and np.all(got[:skew] == 9) and np.all(got[skew + k:] == 9)


def test_too_many_are_refused(scn, ctx):
    p, n = (C.c_void_p * 9)(), (C.c_size_t * 9)()
    assert scn.lib().scn_copy_many(ctx.h, p, p, n, 9) != 0
    n[0] = 4
    assert scn.lib().scn_copy_many(ctx.h, p, p, n, 1) != 0
