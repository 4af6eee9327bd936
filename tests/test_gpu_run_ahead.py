"""A resident batch's layers queued behind its rule books, their numbers of rows read on the device: whatever batches
came before, the probabilities and the multiply-adds are those of a net that has seen no other batch (which waits for
its counts), bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(cfg, weights, fused):
    from sparseconvnet_archived_amd import hostapi
    net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, nTop=1, threads=1)
    cfg.build(net)
    net.setFusedConvolutions(fused)
    for i, (W, B, pr) in (weights or {}).items():
        net.set_weights(i, W, B, pr)
    return net


# (samples of the batches in turn: the bounds hold, are outgrown, and are far too wide; kernels of few rows and of many)
@pytest.mark.parametrize("config,sizes,fused,bf16", [(2, (3, 3, 40, 1, 40, 2), True, False), (2, (30, 30, 5), False, False),
                                                     (2, (8, 9, 60, 7), True, True), (3, (2, 2, 9, 1), True, False)])
def test_layers_ahead_of_the_counts(scn, config, sizes, fused, bf16):
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(config, batch=max(sizes))
    net = _net(cfg, None, fused)
    weights = synthetic.he_normal_weights(net.layers(), 5)
    net.close()
    net = _net(cfg, weights, fused)
    ctx = scn.Context(handle=net.context_handle())
    for i, b in enumerate(sizes):
        S, K, R, bg, feats, n = synthetic.codify(synthetic.make_samples(cfg, 300 + i, batch=b), cfg.dimension, cfg.lattice,
                                                 net.inputSpatialSize, cfg.nInputFeatures)
        got = []
        for use in (net, _net(cfg, weights, fused)):
            use.setPrecision(scn.BF16 if bf16 else scn.FP32)
            d = [ctx.array(S, np.int32), ctx.array(K, np.int64), ctx.array(R, np.int32), ctx.array(bg, np.int32),
                 ctx.array(feats, np.float32)]
            ctx.sync()
            p = np.zeros((b, cfg.nClasses), np.float32)
            hostapi.take_multiply_add_count()
            use.forward_resident(b, d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, len(K), n, d[4].ptr, p)
            got.append((p, hostapi.take_multiply_add_count(), use.interface(2), use.interface(6)))
            if use is not net:
                use.close()
        a, w = got
        assert np.isfinite(a[0]).all() and np.array_equal(a[0], w[0]), (i, b)
        assert a[1] == w[1] > 0, (i, b)
        for x, y in zip(a[2:], w[2:]):
            assert x["nSpatialSites"] == y["nSpatialSites"] and np.array_equal(x["features"], y["features"]), (i, b)
    net.close()
