"""The host view of a batch's grids (SpatiallySparseBatchInterface::downloadGrids), batch after batch, on the CPU: a reset
gives it back, and what the producers keep of an input's grids is no more than a batch has."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "sparseconvnet-archived_amd")


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("grids") / "libbatch_grids.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-I", os.path.join(PKG, "host"),
                           "-I", os.path.join(os.path.dirname(PKG), "include"),
                           os.path.join(HERE, "batch_grids_harness.cpp"), "-o", out, "-L", PKG, "-lscn_host", "-lscn_hip",
                           "-Wl,-rpath," + PKG])
    lib = C.CDLL(out)
    lib.held.argtypes = [C.c_int] * 4 + [C.POINTER(C.c_int)]
    return lib


@pytest.mark.parametrize("batches", [1, 3, 200])
def test_a_reset_gives_the_grids_back(harness, batches):
    most = C.c_int()
    assert harness.held(batches, 20, 50, 0, C.byref(most)) == 0


@pytest.mark.parametrize("batches", [2, 3, 200])
def test_kept_grids_are_no_more_than_a_batch_has(harness, batches):
    most = C.c_int()
    assert harness.held(batches, 20, 50, 1, C.byref(most)) <= 20
    assert 19 <= most.value <= 20
