"""scn_gather_rows of few rules: workgroups of fewer rules, down to between two and four loads a lane, and the bytes are the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rules below and above those of a workgroup a compute unit (256 x 256), one and none over; chunks of one word to 4096; 16 rules
@pytest.mark.parametrize("count,nIn", [(1, 4096), (7, 640), (17, 1020), (33, 96), (1001, 128), (65279, 36), (65281, 36), (4097, 3),
                                       (32769, 64), (600, 2048)])
def test_gather(scn, ctx, count, nIn):
    rng = np.random.default_rng(count)
    x, rules = rng.standard_normal((97, nIn), dtype=np.float32), rng.integers(-1, 97, count).astype(np.int32)
    out = ctx.array(np.full((count + 3, nIn), 7, np.float32))
    ctx.gather_rows(ctx.array(x), out, ctx.array(rules), count, nIn)
    got = out.download()
    assert np.array_equal(got[:count], np.where(rules[:, None] >= 0, x[np.maximum(rules, 0)], 0)) and np.all(got[count:] == 7)
