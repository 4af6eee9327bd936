"""The same with more shared out than such small fields would be, on the CPU under the sanitizer: every level's mask
by several wavefronts, and a sample's rule books by several workgroups, each with some of the layers or with a slab
of one of them (chain_parts_harness.cpp).  The chains, the oracle and the guard words are test_chain_cpu.py's."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import test_chain_cpu as whole

SRC = os.path.join(whole.HERE, "chain_parts_harness.cpp")
LIB = os.path.join(whole.HERE, "libchain_parts_cpu.so")


@pytest.fixture(scope="module")
def harness():
    if not os.path.exists(LIB) or os.path.getmtime(LIB) < max(os.path.getmtime(p)
                                                              for p in (SRC, whole.SRC) + whole.HEADERS):
        subprocess.check_call(["g++", "-O1", "-g", "-std=c++17", "-shared", "-fPIC", "-Wall", "-fsanitize=undefined",
                               "-fno-sanitize-recover=undefined", "-static-libubsan",
                               "-I", whole.CSRC, "-I", whole.HERE, SRC, "-o", LIB])
    lib = C.CDLL(LIB)
    lib.pyr_cpu_chain.restype = C.c_int
    return lib


@pytest.mark.parametrize("parts", (1, 2, 5, 11, 40))
@pytest.mark.parametrize("case", range(len(whole.CHAINS)))
def test_samples_by_parts(harness, case, parts):
    d, n0, layers = whole.CHAINS[case]
    fill = 0.08 if n0 ** d <= 8192 else 0.025
    harness.pyr_cpu_parts(parts)
    for seed, batch, T in ((1, 5, 64), (2, 1, 32)):
        whole.check(harness, d, n0, layers, batch, 100 * case + seed, T=T, fill=fill)
    assert 1 <= harness.pyr_cpu_parts(parts) <= 24


@pytest.mark.parametrize("case", range(len(whole.WINDOWED)))
def test_parts_a_window_at_a_time(harness, case):
    """with little LDS: the rows of the layer before a part come from a window of their own"""
    d, n0, layers, fill = whole.WINDOWED[case]
    for kb in (14, 20, 30, 60):
        for parts in (2, 7, 30):
            harness.pyr_cpu_parts(parts)
            rc, *_ = whole.run_chain(harness, d, n0, layers, 4, 700 + case, fill=fill, lds=kb * 1024, T=64)
            if rc == 0:
                whole.check(harness, d, n0, layers, 4, 700 + case, fill=fill, lds=kb * 1024, T=64)


@pytest.mark.parametrize("seed", range(12))
def test_shapes_of_fields_windows_and_densities(harness, seed):
    """odd strides (windows that leave gaps among them), fields of one to four words a row, empty and full samples"""
    rng = np.random.default_rng(seed)
    for _ in range(4):
        d = int(rng.integers(1, 4))
        sizes = (1, 2, 3, 4) if d == 2 else (1, 2) if d == 3 else (1, 2, 3, 5, 16)
        layers, n = [], int(rng.integers(1, 4))
        for _ in range(int(rng.integers(1, 6))):  # from the output side, so that the windows tile
            size, stride = int(rng.choice(sizes)), int(rng.integers(1, 4))
            if (n - 1) * stride + size > {1: 500, 2: 200, 3: 24}[d]:
                break
            n = (n - 1) * stride + size
            layers.insert(0, ("c", size, stride))
        if not layers:
            continue
        if rng.integers(0, 2):
            layers.append(("t",))
        harness.pyr_cpu_parts(int(rng.integers(1, 25)))
        fill = float(rng.choice([0.01, 0.08, 0.5])) if n ** d <= 4096 else 0.03
        whole.check(harness, d, n, layers, int(rng.integers(1, 6)), 31 * seed, T=64, fill=fill)


def test_layers_were_cut_into_slabs(harness):
    for case in (2, 3, 4):
        d, n0, layers = whole.CHAINS[case]
        harness.pyr_cpu_parts(40)
        whole.check(harness, d, n0, layers, 2, 77, T=64, fill=0.05)
    assert harness.pyr_cpu_parts(-1) >= 3
