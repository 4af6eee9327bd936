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


# no more rows than the kernel of few rows takes and one more, both numbers of row groups; columns in two slices; channels
# in fours and a window beyond the thin kernel's, which are gathered first; images along
@pytest.mark.parametrize("rows", [0, 1, 512, 513, 545, 49153])
@pytest.mark.parametrize("fs,nIn,N", [(8, 1, 32), (4, 3, 36), (4, 7, 260), (2, 4, 32), (27, 1, 30), (32, 1, 32)])
def test_convolution_that_leaves_its_matrix(scn, ctx, rows, fs, nIn, N):
    rng = np.random.default_rng(rows + N)
    K = fs * nIn
    d_in = ctx.array(rng.standard_normal((700, nIn), dtype=np.float32))
    h_rules = rng.integers(-1, 700, (max(rows, 1), fs)).astype(np.int32)
    d_rules = ctx.array(h_rules)
    d_W, d_B = ctx.array(rng.standard_normal((K, N), dtype=np.float32)), ctx.array(rng.standard_normal(N, dtype=np.float32))
    d_other = ctx.array(rng.standard_normal((64, 32), dtype=np.float32))
    matrix, two_matrix = (ctx.array(np.full((rows + 70, K), 7, np.float32)) for _ in range(2))
    one, two = (ctx.array(np.full((rows + 70, N), 7, np.float32)) for _ in range(2))
    now, later = (ctx.array(np.full(64 * 32 * 3 // 2, 7, np.int32)) for _ in range(2))
    print("convolution and its matrix", rows, fs, nIn, N, flush=True)
    ctx.weight_images_many([(d_other, now, 64, 32, 0, scn.FP32_PLANES)])
    ctx.gather_rows(d_in, two_matrix, d_rules, rows * fs, nIn)
    ctx.nin_forward(two_matrix, d_W, d_B, None, two, rows, K, N, 0.5, scn.LEAKYRELU)
    ctx.weight_images_many([(d_other, later, 64, 32, 0, scn.FP32_PLANES)], later=True)
    scn._check(scn.lib().scn_conv_nin_forward_matrix(ctx.h, d_in.ptr, d_rules.ptr, fs, nIn, matrix.ptr, d_W.ptr, d_B.ptr, None,
                                                     one.ptr, rows, N, 0.5, scn.LEAKYRELU, scn.FP32))
    ctx.weight_images_many([], later=True)  # (left where no launch took it: given up before its room goes)
    if rows > 512 and N % 4 == 0 and nIn % 4 and fs <= 27:  # (one launch, which takes the image along)
        assert np.array_equal(now.download(), later.download())
    assert np.array_equal(matrix.download(), two_matrix.download())
    assert np.array_equal(one.download(), two.download())


# one group of rows and two; columns in one slice and in two, of which one makes the images; images of one workgroup and of
# many, of three planes and one; and images that no first layer takes along, made before the layer that is given one
@pytest.mark.parametrize("M,N", [(900, 32), (70001, 160), (600, 300), (0, 32)])
@pytest.mark.parametrize("shapes", [[(64, 32)], [(256, 96), (640, 320), (64, 4)]])
def test_images_beside_a_first_layer(scn, ctx, M, N, shapes):
    rng = np.random.default_rng(M + N)
    items, want = [], []
    for k, (K, n) in enumerate(shapes):
        precision = scn.BF16 if k == 1 else scn.FP32_PLANES
        W = ctx.array(rng.standard_normal((K, n), dtype=np.float32))
        words = K * ((n + 31) // 32 * 32) * (3 if precision == scn.FP32_PLANES else 1) // 2
        now, later = (ctx.array(np.full(words, 7, np.int32)) for _ in range(2))
        ctx.weight_images_many([(W, now, K, n, 0, precision)])
        items.append((W, later, K, n, 0, precision))
        want.append(now)
    x = rng.standard_normal((500, 3), dtype=np.float32)
    rules = rng.integers(-1, 500, (max(M, 1), 4)).astype(np.int32)
    W, B = rng.standard_normal((12, N), dtype=np.float32), rng.standard_normal(N, dtype=np.float32)
    args = ctx.array(x), ctx.array(rules), 4, 3, ctx.array(W), ctx.array(B), None
    one, two = (ctx.array(np.full((M + 8, N), 7, np.float32)) for _ in range(2))
    print("images beside", M, N, shapes, flush=True)
    ctx.conv_nin_forward(*args, one, M, N)
    ctx.weight_images_many(items, later=True)
    ctx.conv_nin_forward(*args, two, M, N)
    assert np.array_equal(one.download(), two.download())
    K, n = shapes[0]
    if M == 0:  # (nothing has been launched: the layer that reads its image has it made)
        A, out = ctx.array(rng.standard_normal((300, K), dtype=np.float32)), [ctx.empty((300, n), np.float32) for _ in range(2)]
        bias = ctx.array(np.zeros(n, np.float32))
        for o, im in zip(out, (want[0], items[0][1])):
            scn._check(scn.lib().scn_conv_nin_forward_image(ctx.h, A.ptr, None, 1, K, items[0][0].ptr, im.ptr, bias.ptr, None, o.ptr,
                                                            300, n, 1.0, scn.NOSIGMOID, scn.FP32_PLANES))
        assert np.array_equal(out[0].download(), out[1].download())
    for now, (_, later, *_) in zip(want, items):
        assert np.array_equal(now.download(), later.download())
