"""Pictures of points on the CPU: points that meet in a site, points outside the field, fields with a bit for every site and
larger ones; and the map of a grid whose entries were appended without its index."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from __graft_entry__ import load_package

load_package()
from sparseconvnet_archived_amd import hostapi  # noqa: E402

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "sparseconvnet-archived_amd")


# 256^3 sites: the most that have bits; 257^3: looked up in the grid's map
@pytest.mark.parametrize("d,lattice,field,n", [(2, 20, 26, 0), (2, 20, 26, 1), (2, 20, 26, 500), (1, 9, 70, 30), (3, 30, 24, 2000),
                                               (3, 250, 256, 300), (3, 250, 257, 300), (3, 40, 40, 5)])
def test_points(d, lattice, field, n):
    rng = np.random.default_rng(lattice + n)
    ds = hostapi.Dataset("points", 3, 2)
    pictures = []
    for _ in range(3):  # (the bits are clean again for the next one)
        at = rng.integers(0, min(lattice, 40), (n, d)).astype(np.int32)
        feats = rng.standard_normal((n, 3), dtype=np.float32)
        ds.add_points(d, lattice, at, feats, 1)
        pictures.append((at, feats))
    for i, (at, feats) in enumerate(pictures):
        k, r, bg, f = ds.codify(i, field)
        shift = int((field - lattice) / 2)
        keys, rows, want = [], [], [np.zeros(3, np.float32)]
        for p, value in zip(at + shift, feats):
            if (p < 0).any() or (p >= field).any():
                continue
            key = 0
            for x in p:
                key = key * field + int(x)
            if key not in keys:
                keys.append(key)
                rows.append(len(want))
                want.append(value)
        assert bg == 0 and np.array_equal(f, np.array(want))
        assert dict(zip(k.tolist(), r.tolist())) == dict(zip(keys, rows))


@pytest.mark.parametrize("n,split", [(0, 0), (1, 0), (1, 1), (40, 0), (40, 17), (1000, 1000), (1000, 1)])
def test_appended_entries_are_found(tmp_path, n, split):
    out = str(tmp_path / "libpoints.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-I", os.path.join(PKG, "host"),
                           os.path.join(HERE, "points_picture_harness.cpp"), "-o", out])
    f = C.CDLL(out).appended
    p64, p32 = C.POINTER(C.c_int64), C.POINTER(C.c_int)
    f.argtypes = [p64, C.c_int, C.c_int, p64, p32]
    keys = np.random.default_rng(n).permutation(5 * n + 1)[:n].astype(np.int64)
    k, r = np.empty(n, np.int64), np.empty(n, np.int32)
    assert f(keys.ctypes.data_as(p64), n, split, k.ctypes.data_as(p64), r.ctypes.data_as(p32)) == 0
    order = np.argsort(keys)
    assert np.array_equal(k, keys[order]) and np.array_equal(r, order)
