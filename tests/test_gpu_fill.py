"""Fills at any alignment."""
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
