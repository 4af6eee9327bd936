"""A new net's first batch: the weights' layouts of all its layers lie in the room that its stream has had from the start,
so that the batch allocates no more than one in a precision that has none."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_no_memory_for_images_in_a_first_batch(scn):
    from sparseconvnet_archived_amd import hostapi, synthetic
    cfg = synthetic.config(4, batch=40)
    samples = synthetic.make_samples(cfg, 9)
    ds = hostapi.Dataset(cfg.name, cfg.nInputFeatures, cfg.nClasses, hostapi.TESTBATCH)
    for pts, f, label in samples:
        ds.add_points(cfg.dimension, cfg.lattice, pts, f, label)
    taken, images = {}, 0
    # (the first net of a process: kernels are loaded)
    for what, precision in (("first", scn.FP32), ("none", scn.BF16X3), ("images", scn.FP32)):
        net = hostapi.Net(cfg.dimension, cfg.nInputFeatures, cfg.nClasses, threads=1)
        cfg.build(net)
        for i, (W, B, pr) in synthetic.he_normal_weights(net.layers(), 2).items():
            net.set_weights(i, W, B, pr)
        net.setPrecision(precision)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        net.begin(ds, len(samples))
        assert net.next_batch()
        torch.cuda.synchronize()
        taken[what] = free - torch.cuda.mem_get_info()[0]
        if what == "images":
            for i, l in enumerate(net.layers()):
                if l["kind"].startswith("nin"):
                    rows = net.interface(i + 1, want_features=False)["nSpatialSites"]
                    images += scn.lib().scn_weight_image_bytes(C.c_void_p(net.context_handle()), rows, l["nIn"], l["nOut"],
                                                               l["nIn"], scn.FP32_PLANES)
        net.end()
        net.close()
    print("taken", taken, "images", images, flush=True)
    assert images >= 8 << 20
    # (in whole pages of 2 MB, of some of the buffers)
    assert taken["images"] <= taken["none"] + (4 << 20)
