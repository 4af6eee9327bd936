"""The end of a net in one launch (scn_terminal_classifier): the mean of the terminal pooling bit for bit the one
scn_terminal_pool gives, probabilities bit for bit those of scn_nin_forward on it, and both against float64."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,S", [(1, 4, 4, 1), (2, 192, 100, 4), (3, 128, 40, 8), (61, 800, 100, 9), (5, 100, 128, 17),
                                     (511, 36, 12, 3), (512, 1024, 20, 2), (7, 1020, 100, 70)])
def test_terminal_classifier(scn, ctx, M, K, N, S):
    print("terminal classifier", M, K, N, S, flush=True)
    rng = np.random.default_rng(M + K)
    nIn = 2 * M * S
    x = rng.standard_normal((nIn, K)).astype(np.float32)
    rules = rng.integers(0, nIn, (M, S)).astype(np.int32)
    for b in range(M):  # samples of one row up to the batch's most
        rules[b, rng.integers(1, S + 1):] = -1
    rules[-1] = rng.integers(0, nIn, S)
    W = (rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32)
    B = rng.uniform(-0.5, 0.5, N).astype(np.float32)
    d_x, d_rules, d_W, d_B = (ctx.array(a) for a in (x, rules, W, B))
    pooled, probs, copy = (ctx.array(np.full(s, 7, np.float32)) for s in ((M, K), (M, N), (M, N)))
    pooled2, probs2 = ctx.empty((M, K), np.float32), ctx.empty((M, N), np.float32)
    assert scn.lib().scn_terminal_classifier_supported(M, K, N)
    for target in (copy, None):
        ctx.terminal_classifier(d_x, d_rules, M, S, pooled, d_W, d_B, probs, target, K, N, 0.75)
        ctx.terminal_pool(d_x, pooled2, d_rules, M, S, K)
        ctx.nin_forward(pooled2, d_W, d_B, None, probs2, M, K, N, 0.75, scn.SOFTMAX, scn.FP32_PLANES)
        assert np.array_equal(pooled.download(), pooled2.download())
        assert np.array_equal(probs.download(), probs2.download())
    assert np.array_equal(copy.download(), probs.download())
    assert np.array_equal(pooled.download(), orc.terminal_pool(x, rules, M, S, K))
    z = 0.75 * (pooled.download().astype(np.float64) @ W.astype(np.float64) + B)
    e = np.exp(z - z.max(1, keepdims=True))
    # (a sum of K products of fp32: its rounding is below K / 2 of 2^-24 of the terms, in the exponent of the soft-max)
    bound = 1e-6 + K / 2.0 * 2.0 ** -24 * (np.abs(pooled.download()) @ np.abs(W)).max()
    assert np.abs(probs.download() - e / e.sum(1, keepdims=True)).max() <= bound


def test_shapes_it_does_not_take(scn, ctx):
    lib = scn.lib()
    for M, K, N in ((0, 64, 100), (513, 64, 100), (8, 1028, 100), (8, 66, 100), (8, 64, 10), (8, 64, 132), (8, 64, 96)):
        assert not lib.scn_terminal_classifier_supported(M, K, N)
        assert lib.scn_terminal_classifier(ctx.h, None, None, M, 1, None, None, None, None, None, K, N, 1.0) != 0


def test_the_last_launch_has_a_row_of_its_own_in_a_profile(scn):
    """a net's spans by family and layer: the terminal pooling and the classifier in one, under the classifier"""
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(2, batch=3)
    net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, threads=1)
    cfg.build(net)
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TESTBATCH)
    for pts, f, label in synthetic.make_samples(cfg, 5):
        ds.add_points(cfg.dimension, cfg.lattice, pts, f, label)
    c = scn.Context(handle=net.context_handle())
    c.prof_enable(True)
    net.begin(ds, cfg.batch)
    assert net.next_batch()
    net.end()
    rows = [(fam, tag) for fam, tag, _ in c.prof_spans() if tag >= len(net.layers()) - 2]
    c.prof_enable(False)
    assert net.layers()[-2]["kind"] == "terminal" and rows == [("net_end", len(net.layers()) - 1)], rows


def test_the_launch_for_all_layers_weights_has_no_layer_in_a_profile(scn):
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(2, batch=40)
    net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, threads=1)
    cfg.build(net)
    net.setFusedConvolutions(True)
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TESTBATCH)
    for pts, f, label in 2 * synthetic.make_samples(cfg, 5):
        ds.add_points(cfg.dimension, cfg.lattice, pts, f, label)
    c = scn.Context(handle=net.context_handle())
    c.prof_enable(True)
    net.begin(ds, cfg.batch)
    assert net.next_batch() and net.next_batch()
    net.end()
    nin = [tag for fam, tag, _ in c.prof_spans() if fam == "nin"]
    c.prof_enable(False)
    # (the layer without a convolution, and the weights; the classifier's launch is the net's end)
    assert sorted(nin) == [-1, -1, len(net.layers()) - 3, len(net.layers()) - 3], nin
