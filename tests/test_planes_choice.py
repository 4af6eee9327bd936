"""The choice of a contraction's tile, costed as it is launched, and of the weight gradients' tiles and of those that share a launch, on the CPU."""
import ctypes as C
import math
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "sparseconvnet-archived_amd", "csrc")
# of the tiles of which a workgroup may take several, three planes: rows, columns, fewest blocks of 32 k that are several tiles to a
# workgroup; microseconds of a tile alone and of its block, and of several: of them all, of each and of its block
TILES = {0: (128, 128, 2, 4.1, 1.04, 2.5, 2.1, 1.12), 1: (256, 64, 2, 4.3, 1.25, 1.6, 3., 1.3),
         3: (64, 128, 3, 3.4, .68, 3.1, 1.45, .71)}


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("choice") / "libchoice.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-I", CSRC,
                           os.path.join(HERE, "planes_choice_harness.cpp"), "-o", out])
    lib = C.CDLL(out)
    lib.lines_tile.argtypes = [C.c_int, C.c_int, C.c_int64, C.c_int, C.c_int, C.c_int]
    lib.lines_tile_cost.argtypes = [C.c_int, C.c_int, C.c_int, C.c_int64, C.c_int, C.c_int, C.c_int]
    lib.lines_tile_cost.restype = C.c_float
    lib.lines_tile_long.argtypes = [C.c_int, C.c_int, C.c_int64, C.c_int, C.c_int]
    return lib


# plain rows of less than their weights (the image 6 N K bytes, the rows 4 M K) are launched a workgroup a tile, others several
# tiles to a workgroup; one row more or fewer at the line between the two
@pytest.mark.parametrize("M,K,N", [(3000, 512, 3008), (2500, 256, 2048), (2600, 1024, 1920), (2880, 128, 1920), (2879, 128, 1920),
                                   (139000, 384, 128), (40000, 96, 640), (9001, 64, 804), (5000, 64, 4096), (70000, 32, 96),
                                   (70000, 512, 64), (70000, 544, 64)])
def test_a_tile_costs_what_its_launch_does(choice, M, K, N):
    for t, (rows, columns, least, f, t1, begin, each, block) in TILES.items():
        wgs, per, T = -(-M // rows) * -(-N // columns), choice.lines_tile_long(256, t, M, K, N), K // 32
        if wgs <= 256:
            assert per == 0
            continue
        assert (per > 0) == (-(-N // 32) * 32 * 6 <= 4 * M and least <= T <= 16 and -(-N // columns) <= 32)
        n = wgs / 256
        want = (begin + -(-wgs // (8 * per)) * (each + T * block) if per else
                (math.ceil(n) if n <= 3 else n + .5) * (f + T * t1))
        assert choice.lines_tile_cost(256, 3, t, M, K, N, 0) == pytest.approx(want, rel=1e-5), t


# measured: 28.0 us in the tile of 64 x 128 and 25.0 in this; 77 and 68
@pytest.mark.parametrize("M,K,N", [(2500, 256, 2048), (2600, 1024, 1920)])
def test_rows_of_less_than_their_weights(choice, M, K, N):
    assert choice.lines_tile(256, 3, M, K, N, 0) == 2


# measured in every tile: the 64 x 64 of which two share a compute unit 19.0 and 46.4 us, several tiles of the others to a
# workgroup no less than 20.4 and 52.5
@pytest.mark.parametrize("M,K,N", [(70000, 160, 36), (70000, 512, 64)])
def test_rows_of_few_columns(choice, M, K, N):
    assert choice.lines_tile(256, 3, M, K, N, 0) == 4


def test_shapes_of_several_tiles_to_a_workgroup(choice):
    """those of the tests on the card are launched so, in all the tiles that can be"""
    from test_gpu_lines import SEVERAL
    tiles = [choice.lines_tile(256, 3, M, K, N, 0) for M, K, N in SEVERAL]
    assert all(choice.lines_tile_long(256, t, *s) > 0 for t, s in zip(tiles, SEVERAL)) and set(tiles) == set(TILES)


# measured with the pooling behind it: 100000 x 96 x 192 76 us past the caches and 65 through them, 600000 x 64 x 64 145 and 158
@pytest.mark.parametrize("M,K,N,gradient,want", [(100000, 96, 192, 0, 0), (100000, 96, 192, 1, 1), (600000, 64, 64, 0, 1),
                                                 (1 << 19, 64, 64, 0, 0), ((1 << 19) + 1, 64, 64, 0, 1)])
def test_results_past_the_caches(choice, M, K, N, gradient, want):
    choice.past_caches.argtypes = [C.c_int64, C.c_int, C.c_int, C.c_int]
    assert choice.past_caches(M, K, N, gradient) == want


SMALL, FIRST, LARGE, EMPTY, OTHER = ((11400, 384, 128, 2, 25), (83597, 12, 32, 1, 21), (139000, 384, 128, 2, 25), (0, 384, 128, 2, 25),
                                     (5000, 30, 7, 0, 25))


# (one alone: 23.5 us in the launch for several, 15.7 by itself)
@pytest.mark.parametrize("items,want", [([], []), ([SMALL], [0]), ([FIRST], [0]), ([SMALL, FIRST], [1, 1]), ([LARGE, SMALL], [0, 0]),
                                        ([SMALL, EMPTY, OTHER], [0, 0, 0]), ([SMALL, LARGE, FIRST, EMPTY], [1, 0, 1, 0]),
                                        ([SMALL] * 24, [1] * 24)])
def test_weight_gradients_of_one_launch(choice, items, want):
    columns = [(C.c_int64 if i == 0 else C.c_int) * max(1, len(items)) for i in range(5)]
    out = (C.c_int * max(1, len(items)))()
    assert choice.joined(256, len(items), *(t(*(x[i] for x in items)) for i, t in enumerate(columns)), out) == sum(want)
    assert list(out)[:len(items)] == want


# (wavefronts of sixteen rows, microseconds a step of them all and of a range, rows loaded into registers and by lines)
ATB = [(1, 1, (8, 8), (.8, .67), (4., 2.2)), (2, 1, (8, 12), (1.13, 1.4), (4., 3.7)), (1, 2, (8, 12), (1.13, 1.42), (4., 4.2)),
       (2, 2, (8, 8), (1.95, 1.36), (6., 3.7))]


@pytest.mark.parametrize("M", [1, 127, 129, 193, 1000, 3000, 45000, 139000])
@pytest.mark.parametrize("K,N", [(32, 32), (12, 32), (384, 128), (864, 64), (1280, 480)])
@pytest.mark.parametrize("lines,pairsA,pairsD,twoByTwo", [(1, 1, 1, 1), (1, 1, 1, 0), (0, 0, 1, 0), (0, 0, 0, 1)])
def test_a_weight_gradient_costs_what_its_launch_does(choice, M, K, N, lines, pairsA, pairsD, twoByTwo):
    """ranges are whole steps of the workgroup that takes them, as many as are costed, and none of the other tiles with any
    number of ranges up to 64 costs less"""
    rows, cost = C.c_int64(), C.c_double()
    choice.atb.argtypes = [C.c_int, C.c_int64] + 6 * [C.c_int] + [C.POINTER(C.c_int64), C.POINTER(C.c_double)]
    tile = choice.atb(256, M, K, N, lines, pairsA, pairsD, twoByTwo, rows, cost)

    def costs(t, rows):
        mt, nt, waves, ti, f = ATB[t]
        tiles, ranges = -(-K // (32 * mt)) * -(-N // (32 * nt)), -(-M // rows)
        return (-(-tiles * ranges // 256) * (rows // (16 * waves[lines]) * ti[lines] + f[lines]) + tiles * ranges * mt * nt * 1024 / 2e5)

    allowed = [t for t, (mt, nt, *_) in enumerate(ATB) if (t < 3 or twoByTwo) and (mt == 1 or pairsA) and (nt == 1 or pairsD)]
    assert tile in allowed and rows.value > 0 and rows.value % (16 * ATB[tile][2][lines]) == 0
    assert cost.value == pytest.approx(costs(tile, rows.value))
    for t in allowed:
        each = 16 * ATB[t][2][lines]
        for s in range(1, min(64, -(-M // each)) + 1):
            if -(-K // (32 * ATB[t][0])) * -(-N // (32 * ATB[t][1])) * s <= 8 * 256:
                assert cost.value <= costs(t, -(-M // (s * each)) * each) * (1 + 1e-9)
