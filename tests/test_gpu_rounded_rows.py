"""Rows that a pooling leaves rounded to bf16 beside its output: the contraction's bits are those of fp32 rows, which it
rounds itself, in every kernel that takes them."""
import numpy as np
import pytest

from test_gpu_capture import Graph

pytestmark = pytest.mark.gpu


def rounded(v):  # to the nearest bf16, ties to the even one
    u = np.ascontiguousarray(v, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7fff + (u >> 16 & 1)) >> 16).astype(np.uint16)


@pytest.mark.parametrize("rows,out,ps,C", [(300, 1, 4, 8), (3000, 777, 9, 32), (500, 2000, 8, 160), (900, 63, 5, 12)])
def test_the_pooling_rounds(scn, ctx, rows, out, ps, C):
    rng = np.random.default_rng(C)
    d_in, rules = ctx.array(rng.standard_normal((rows, C), dtype=np.float32)), rng.integers(-1, rows, (out, ps)).astype(np.int32)
    d_rules = ctx.array(rules)
    a, b = [(ctx.array(np.full((out + 5, C), 7, np.float32)), ctx.array(np.full((out + 5, C), 7, np.int32))) for _ in range(2)]
    d16 = ctx.array(np.full((out + 5, C // 2), 7, np.int32))
    ctx.maxpool(d_in, a[0], d_rules, out, ps, C, a[1])
    ctx.maxpool_rounded(d_in, rows, b[0], d16, d_rules, out, ps, C, b[1])
    got = b[0].download()
    assert np.array_equal(a[0].download(), got) and np.array_equal(a[1].download(), b[1].download())
    half = d16.download()
    assert np.array_equal(half[:out].view(np.uint16).reshape(out, C), rounded(got[:out])) and np.all(half[out:] == 7)
    assert scn.lib().scn_maxpool_rounded(ctx.h, d_in.ptr, rows, b[0].ptr, d16.ptr, d_rules.ptr, out, ps, 6, b[1].ptr) != 0


# (rows, fs, nIn, N) few rows, by the split contractions, by lines, by rings of a wavefront's own; long ones of few rows
@pytest.mark.parametrize("rows,fs,nIn,N", [(40, 4, 64, 96), (900, 4, 320, 480), (26000, 4, 160, 320), (41600, 4, 64, 96), (10500, 4, 480, 640),
                                           (6001, 4, 384, 256), (20003, 27, 64, 128), (9000, 8, 32, 64)])
def test_the_bits_of_fp32_rows(scn, ctx, rows, fs, nIn, N):
    rng = np.random.default_rng(rows)
    K, n = fs * nIn, 1200
    x = rng.standard_normal((n, nIn), dtype=np.float32)
    d_x, d_x16 = ctx.array(x), ctx.array(rounded(x).view(np.int32))
    d_rules = ctx.array(rng.integers(-1, n, (rows, fs)).astype(np.int32))
    d_W = ctx.array((rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32))
    d_B, d_slopes = (ctx.array(rng.uniform(0.1, 0.4, N).astype(np.float32)) for _ in range(2))
    image, room = ctx.empty((-(-N // 32) * 32 * K * 2 // 4,), np.float32), ctx.empty((n, nIn // 2), np.float32)
    ctx.weight_images_many([(d_W, image, K, N, 0, scn.BF16)])
    outs = [ctx.array(np.full((rows + 300, N), 7, np.float32)) for _ in range(5)]
    print("rounded rows", rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward(d_x, d_rules, fs, nIn, d_W, d_B, d_slopes, outs[0], rows, N, 1.0, scn.PRELU, scn.BF16)
    ctx.conv_nin_forward_rounded(d_x, d_x16, d_rules, fs, nIn, d_W, image, d_B, d_slopes, outs[1], rows, N, 1.0, scn.PRELU)
    ctx.conv_nin_forward_rounded(d_x, d_x16, d_rules, fs, nIn, d_W, None, d_B, d_slopes, outs[2], rows, N, 1.0, scn.PRELU)
    ctx.conv_nin_forward_a16(d_x, n, room, d_rules, fs, nIn, d_W, d_B, d_slopes, outs[3], rows, N, 1.0, scn.PRELU)
    with Graph(ctx) as g:
        ctx.conv_nin_forward_rounded(d_x, d_x16, d_rules, fs, nIn, d_W, image, d_B, d_slopes, outs[4], rows, N, 1.0, scn.PRELU)
    for _ in range(2):
        g.replay(ctx)
    got = [o.download() for o in outs]
    g.close()
    assert all(np.array_equal(o, got[0]) and np.all(o[rows:] == 7) for o in got)


def test_a_net_of_bf16_operands(scn):
    """batches whose convolutions read rounded rows, and a small one whose do not: the bits of the pass that gathers"""
    from perf import cases
    runs = []
    for fused in (False, True):
        case = dict(name="wide", kind="net", stack="wide", batch=70, precision="bf16", fused=fused)
        s = cases.prepare(case, 3)
        out = [cases.run(s).copy() for _ in range(3)]
        assert all(np.array_equal(o, out[0]) for o in out)
        small = cases._prepare_net(dict(case, batch=2), 4)
        runs.append(np.concatenate([out[0], cases._run_net(small).copy()]))
    assert np.isfinite(runs[0]).all() and np.array_equal(runs[0], runs[1])
