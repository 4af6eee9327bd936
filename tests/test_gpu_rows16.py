"""Long contractions of bf16 rows through rules (k_nin_rows16): the bits of the kernels that a captured call takes, which
has no image of the weights, and nothing stored past the last row."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from test_gpu_capture import Graph

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "sparseconvnet-archived_amd", "csrc")

# (rows, fs, nIn, N, tiles of columns): one to 27 positions in and out of fours, channels of one block of 32 and of several,
# two blocks in all (fewer than the rings hold), a row more than whole workgroups, a slice with tiles past the columns
SHAPES = [(262145, 2, 32, 64, 2), (262399, 4, 32, 96, 3), (262401, 1, 64, 320, 4), (131073, 27, 64, 64, 2), (262337, 27, 32, 64, 2),
          (52225, 27, 64, 96, 3), (26500, 27, 96, 128, 4), (30001, 9, 320, 288, 3), (26625, 8, 128, 160, 3), (52300, 5, 192, 224, 4)]


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    where = tmp_path_factory.mktemp("rows16")
    (where / "choice.cpp").write_text('#include "scn_planes_choice.h"\n'
                                      'extern "C" int tiles(int numCU, long long M, int K, int N) { return rows16_tiles(numCU, M, K, N); }\n')
    out = str(where / "libchoice.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(where / "choice.cpp"), "-o", out])
    lib = C.CDLL(out)
    lib.tiles.argtypes = [C.c_int, C.c_longlong, C.c_int, C.c_int]
    return lib


@pytest.mark.parametrize("rows,fs,nIn,N,tiles", SHAPES)
def test_which_calls_take_it(choice, rows, fs, nIn, N, tiles):
    assert choice.tiles(256, rows, fs * nIn, N) == tiles
    assert choice.tiles(256, rows // 8, fs * nIn, N) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("rows,fs,nIn,N,tiles", SHAPES)
def test_the_same_bits(scn, ctx, rows, fs, nIn, N, tiles):
    rng = np.random.default_rng(rows)
    K = fs * nIn
    d_in, d_in16 = ctx.array(rng.standard_normal((900, nIn), dtype=np.float32)), ctx.empty((900, nIn), np.float32)
    d_rules = ctx.array(rng.integers(-1, 900, (rows, fs)).astype(np.int32))
    d_W = ctx.array((rng.standard_normal((K, N)) * np.sqrt(2.0 / K)).astype(np.float32))
    d_B, d_slopes = (ctx.array(rng.uniform(0.1, 0.4, N).astype(np.float32)) for _ in range(2))
    one, two = (ctx.array(np.full((rows + 256, N), 7, np.float32)) for _ in range(2))
    print("rows16", rows, fs, nIn, N, flush=True)
    ctx.conv_nin_forward_a16(d_in, 900, d_in16, d_rules, fs, nIn, d_W, d_B, d_slopes, one, rows, N, 1.0, scn.PRELU)
    with Graph(ctx) as g:
        ctx.conv_nin_forward_a16(d_in, 900, d_in16, d_rules, fs, nIn, d_W, d_B, d_slopes, two, rows, N, 1.0, scn.PRELU)
    g.replay(ctx)
    got, want = one.download(), two.download()
    g.close()
    assert np.all(got[rows:] == 7) and np.isfinite(got).all() and np.array_equal(got, want)
