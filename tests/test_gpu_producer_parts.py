"""Batches whose pictures several producer threads code in parts: sample for sample what one thread gives."""
import numpy as np
import pytest

from gpu_util import assert_nll

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


def net_of(cfg, threads):
    from sparseconvnet_archived_amd import hostapi, synthetic
    net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, nTop=1, threads=threads)
    cfg.build(net)
    net.setFusedConvolutions(True)
    for i, (W, B, pr) in synthetic.he_normal_weights(net.layers(), 78).items():
        net.set_weights(i, W, B, pr)
    return net


def dataset(cfg, samples, kind=None):
    from sparseconvnet_archived_amd import hostapi
    ds = hostapi.Dataset("parts", 3, 100, hostapi.TESTBATCH if kind is None else kind)
    for at, f, label in samples:
        ds.add_points(2, cfg.lattice, at, f, label)
    return ds


def whole_pass(net, ds, batch):
    """-> probabilities, mistakes and cost of every batch"""
    probs, costs = [], []
    net.begin(ds, batch)
    while net.next_batch():
        out = net.batch_outputs()
        assert out["sampleNumbers"].tolist() == list(range(len(probs), len(probs) + out["batchSize"]))
        probs.extend(out["probabilities"])
        costs.append((out["mistakes"], out["nll"]))  # (by the labels)
    net.end()
    return np.array(probs), costs


def test_constants_for_the_inputs(scn):
    """found over all batches and multiplied into every part's features"""
    from sparseconvnet_archived_amd import synthetic
    cfg = synthetic.config(2, batch=15)
    samples = [(at, f * np.float32([1, 30, 0.02]), label) for at, f, label in pictures(cfg, 31, 60, np.random.default_rng(4))]
    first = None
    for threads in (1, 3, 10):
        net, ds = net_of(cfg, threads), dataset(cfg, samples)
        before = whole_pass(net, ds, 15)[0]
        constants = net.calculateInputRegularizingConstants(ds)
        probs, costs = whole_pass(net, ds, 15)
        net.close()
        first = first or (before, constants, probs, costs)
        assert constants.shape == (3,) and np.all(constants > 0) and not np.array_equal(before, probs)
        assert np.array_equal(first[0], before) and np.array_equal(first[1], constants)
        assert np.array_equal(first[2], probs) and first[3] == costs


@pytest.mark.parametrize("threads", [3, 10])
def test_shuffled_training(scn, threads):
    """A pass at learning rate 0: every sample once, in another order than the dataset's, with its own picture and label."""
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(2, batch=15)
    samples = pictures(cfg, 73, 60, np.random.default_rng(6))
    net = net_of(cfg, 1)
    want = whole_pass(net, dataset(cfg, samples), 15)[0]
    net.close()
    net, ds = net_of(cfg, threads), dataset(cfg, samples, hostapi.TRAINBATCH)
    net.set_training(0.0, 0.0, shuffle=True)
    for _ in range(2):
        order = []
        net.begin(ds, 15)
        while net.next_batch():
            out = net.batch_outputs()
            at = out["sampleNumbers"]
            labels = np.array([samples[i][2] for i in at])
            order += at.tolist()
            # (rows of other batches: other kernels' orders of the sums)
            assert np.allclose(out["probabilities"], want[at], rtol=1e-4, atol=1e-7)
            assert_nll(out["nll"], out["probabilities"].astype(np.float64), labels)
            assert out["mistakes"] == np.sum(out["predictions"][:, 0] != labels)
        net.end()
        assert sorted(order) == list(range(73)) and order != list(range(73))
    net.close()


def test_a_pass_that_is_given_up(scn):
    """with parts of several batches coded or under way; the slots' next pass is whole"""
    from sparseconvnet_archived_amd import synthetic
    cfg = synthetic.config(2, batch=6)
    samples = pictures(cfg, 90, 300, np.random.default_rng(8))
    net = net_of(cfg, 1)
    want = whole_pass(net, dataset(cfg, samples), 6)
    net.close()
    net, ds = net_of(cfg, 4), dataset(cfg, samples)
    for batches in (0, 1, 3, 5):
        net.begin(ds, 6)
        for _ in range(batches):
            assert net.next_batch()
        net.end()
        probs, costs = whole_pass(net, ds, 6)
        assert np.array_equal(want[0], probs) and want[1] == costs
    net.close()
