"""Batches whose pictures several producer threads code in parts: sample for sample what one thread gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pictures(cfg, n, points, rng):
    """points in any order, some of them twice with other features, some outside the field, some pictures without one"""
    out = []
    for i in range(n):
        k = 0 if i % 7 == 3 else int(rng.integers(1, points))
        at = rng.integers(-2 if i % 5 == 1 else 0, cfg.lattice, (k, 2)).astype(np.int32)
        if i % 5 == 1 and k:
            at[0] -= 10 * cfg.lattice
        out.append((at, rng.standard_normal((k, 3), dtype=np.float32), int(rng.integers(0, 100))))
    return out


# (batches smaller than the threads; a last batch of one; one read over the bus, 1 MB, and one copied first, 6 MB)
@pytest.mark.parametrize("n,points,batch", [(9, 60, 1), (23, 60, 2), (31, 60, 15), (90, 700, 90), (330, 1400, 330)])
def test_threads_do_not_matter(scn, n, points, batch):
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(2, batch=batch)
    samples = pictures(cfg, n, points, np.random.default_rng(n))
    results = []
    for threads in (1, 3, 10):
        net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, nTop=1, threads=threads)
        cfg.build(net)
        net.setFusedConvolutions(True)
        for i, (W, B, pr) in synthetic.he_normal_weights(net.layers(), 78).items():
            net.set_weights(i, W, B, pr)
        ds = hostapi.Dataset("parts", 3, 100, hostapi.TESTBATCH)
        for at, f, label in samples:
            ds.add_points(2, cfg.lattice, at, f, label)
        for _ in range(2):  # (the slots' buffers are kept)
            probs, costs = [], []
            net.begin(ds, batch)
            while net.next_batch():
                out = net.batch_outputs()
                assert out["sampleNumbers"].tolist() == list(range(len(probs), len(probs) + out["batchSize"]))
                probs.extend(out["probabilities"])
                costs.append((out["mistakes"], out["nll"]))  # (by the labels)
            net.end()
            results.append((np.array(probs), costs))
        net.close()
    assert results[0][0].shape == (n, 100)
    for probs, costs in results[1:]:
        assert np.array_equal(results[0][0], probs) and results[0][1] == costs
