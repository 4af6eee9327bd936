"""Convolutions over one to three channels through the rules: the bits of the gathered matrix's kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [513, 543, 545, 49152, 49153, 50001])  # (both numbers of row groups, ragged ones)
@pytest.mark.parametrize("fs,nIn,N", [(4, 1, 4), (4, 3, 32), (8, 3, 36), (4, 7, 260)])
def test_thin_convolution(scn, ctx, rows, fs, nIn, N):
    rng = np.random.default_rng(rows + N)
    K = fs * nIn
    d_in = ctx.array(rng.standard_normal((700, nIn), dtype=np.float32))
    h_rules = rng.integers(-1, 700, (rows, fs)).astype(np.int32)
    d_rules = ctx.array(h_rules)
    d_W = ctx.array(rng.standard_normal((K, N), dtype=np.float32))
    d_B = ctx.array(rng.standard_normal(N, dtype=np.float32))
    one, two = (ctx.array(np.full((rows + 70, N), 7, np.float32)) for _ in range(2))
    print("thin convolution", rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward(d_in, d_rules, fs, nIn, d_W, d_B, None, one, rows, N, 1.0, scn.LEAKYRELU)
    m = d_in.download()[h_rules]
    m[h_rules < 0] = 0
    ctx.nin_forward(ctx.array(m.reshape(rows, K)), d_W, d_B, None, two, rows, K, N, 1.0, scn.LEAKYRELU)
    got, want = one.download(), two.download()
    assert np.all(got[rows:] == 7)
    assert np.array_equal(got, want)
