"""Results of batches of changing sizes through one net, whose vectors are written over: the probabilities, predictions
and counts are those of nets that have seen no other batch, for one prediction a sample and for several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ranked(p, k):
    """the k best classes of every row, best first, the lower one ahead where two are as likely"""
    return np.argsort(-p, axis=1, kind="stable")[:, :k].astype(np.int32)


@pytest.mark.parametrize("nTop", [1, 2, 5])
def test_results_of_batches_in_turn(scn, nTop):
    from sparseconvnet_archived_amd import hostapi, synthetic
    sizes = (4, 9, 1, 9, 2)
    cfg = synthetic.config(2, batch=max(sizes))
    net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, nTop=nTop, threads=1)
    cfg.build(net)
    for i, (W, B, pr) in synthetic.he_normal_weights(net.layers(), 5).items():
        net.set_weights(i, W, B, pr)
    ctx = scn.Context(handle=net.context_handle())
    for i, b in enumerate(sizes):
        S, K, R, bg, feats, n = synthetic.codify(synthetic.make_samples(cfg, 400 + i, batch=b), cfg.dimension, cfg.lattice,
                                                 net.inputSpatialSize, cfg.nInputFeatures)
        d = [ctx.array(a, t) for a, t in ((S, np.int32), (K, np.int64), (R, np.int32), (bg, np.int32), (feats, np.float32))]
        ctx.sync()
        p = np.full((b, cfg.nClasses), 7, np.float32)
        print("results", nTop, b, flush=True)
        net.forward_resident(b, d[0].ptr, d[1].ptr, d[2].ptr, d[3].ptr, len(K), n, d[4].ptr, p)
        pred = np.full((b + 1, nTop), -1, np.int32)
        again = np.full((b + 1, cfg.nClasses), 7, np.float32)
        hostapi.lib().scnh_batch_predictions(net.h, hostapi._p(pred))
        hostapi.lib().scnh_batch_probabilities(net.h, hostapi._p(again))
        assert np.allclose(p.sum(1), 1, atol=1e-5)
        assert np.array_equal(again[:b], p) and np.all(again[b] == 7) and np.all(pred[b] == -1)
        assert np.array_equal(pred[:b], _ranked(p, nTop))
    net.close()
