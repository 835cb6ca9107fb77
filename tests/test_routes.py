"""What a call runs as, asked of the library's own choice without a GPU (nk_hip_planned_tile)."""
import ctypes
import random
import time

import numpy as np
import pytest

import numkong_amd as nk
from tests.support import CODES, DIMENSIONS_PER_VALUE, METRICS, STORAGE, STRIPS, route_of

COMPUTE_UNITS = 256  # what the library takes where it cannot ask a device


def strips_of(m, n, stages=2, config=STRIPS):
    return route_of("i8", "dots", m, n, 128 * stages, config)


def walked(m, n, rows, strip_tiles):
    """Tiles that the rounds of resident workgroups walk, one for starting and ending each strip included."""
    strips = -(-(-(-n // 256)) // strip_tiles)
    return -(-(-(-m // rows) * strips) // COMPUTE_UNITS) * (strip_tiles + 1)


# The number of strips against every other number that there is, rows of 128 (2 stages) and of 64 (8).
def test_no_number_of_strips_walks_less():
    rng = random.Random(3)
    for _ in range(300):
        stages = rng.choice((2, 8))
        m, n = int(10 ** rng.uniform(1.9, 5)), int(10 ** rng.uniform(2.2, 5.5))
        rows, route = 128 if stages == 2 else 64, strips_of(m, n, stages)
        assert route.shape == STRIPS and 1 <= route.strip_tiles <= -(-n // 256)
        assert route.units == -(-m // rows) * -(-(-(-n // 256)) // route.strip_tiles)
        tiles = -(-n // 256)
        least = min(walked(m, n, rows, length) for length in range(1, tiles + 1))
        assert walked(m, n, rows, route.strip_tiles) <= 1.06 * least, (m, n, stages) # (of the numbers the eight candidates leave out)


# Planning is part of the call: one with few rows took 2.8 us for it, more than some of them gain from the strips.
def test_planning_takes_no_time():
    def least(shape, config):
        best = 1e9
        for _ in range(30):
            begin = time.perf_counter()
            for _ in range(20):
                route_of("i8", "dots", *shape, config)
            best = min(best, (time.perf_counter() - begin) / 20)
        return best

    tiles, strips = least((100, 300_001, 256), 4), least((100, 300_001, 256), STRIPS)
    assert strips < tiles + 1.0e-6, f"{(strips - tiles) * 1e6:.2f} us more than for a fixed tile"


# Products for which strips were once chosen and took 1.1 to 2 times as long as the tiles that had them before: rows of C of a few
# tiles, strips of three, long rows that start on lines anyway, deep products of integers into rows on the memory's sectors, two
# strips of 64 rows where one tile holds all rows, two stages into a C that the last-level cache takes in, 4-bit types with an image
# that it does not.
@pytest.mark.parametrize("dtype, metric, m, n, k", [
    ("i8", "dots", 1_000_000, 130, 768), ("i8", "angular", 1_000_000, 130, 768), ("bf16", "dots", 200_000, 129, 768), ("u8", "angular", 50_000, 600, 300),
    ("e4m3", "angular", 40_000, 1001, 256), ("u8", "dots", 714, 25_854, 198), ("bf16", "dots", 3340, 6513, 64), ("i8", "euclidean", 349_434, 448, 64),
    ("i8", "euclidean", 6718, 20_000, 448), ("u4", "dots", 947, 85_152, 64), ("i4", "dots", 3276, 27_600, 1920), ("u1", "dots", 25_065, 4016, 896),
    ("u8", "angular", 109, 242_980, 1792), ("u1", "dots", 135, 138_111, 98), ("u1", "dots", 8733, 2341, 18), ("i4", "dots", 5384, 4087, 212), ("bf16", "dots", 5377, 4053, 29),
    ("u4", "dots", 1239, 188_257, 1567), ("u4", "dots", 793, 137_216, 317), ("u4", "dots", 161, 1_191_936, 75), ("u1", "dots", 640, 212_864, 55),
    ("i8", "dots", 2876, 15_004, 1500)])
def test_no_strips_where_they_do_not_pay(dtype, metric, m, n, k):
    assert route_of(dtype, metric, m, n, k).shape != STRIPS


# ... and those that they are for.
@pytest.mark.parametrize("dtype, metric, m, n, k", [
    ("u8", "euclidean", 1000, 500_009, 301), ("f16", "dots", 8192, 8191, 1000), ("i8", "dots", 1024, 204_801, 220), ("bf16", "dots", 527, 400_384, 192),
    ("i8", "angular", 30_000, 2301, 128), ("bf16", "euclidean", 63_086, 5932, 128), ("u8", "angular", 1025, 279_648, 1500), ("e4m3", "dots", 407, 580_128, 340), ("e2m3", "angular", 14_922, 18_880, 2041),
    ("u4", "angular", 17_068, 14_720, 2000), ("e2m3", "dots", 15_185, 15_248, 1325), ("u8", "angular", 14_922, 18_880, 2041)])
def test_strips_where_they_pay(dtype, metric, m, n, k):
    route = route_of(dtype, metric, m, n, k)
    assert route.shape == STRIPS and route.strip_tiles >= 4


# Strips of three tiles where a tile has more to do besides its columns; they were left out with the others for a while, at up to
# 2.7 times the time.
@pytest.mark.parametrize("dtype, metric, m, n, k", [("e2m3", "dots", 2038, 10_937, 77), ("i8", "angular", 1219, 13_997, 179), ("u4", "angular", 436, 39_391, 122), ("bf16", "euclidean", 500, 35_913, 91)])
def test_short_strips(dtype, metric, m, n, k):
    route = route_of(dtype, metric, m, n, k)
    assert route.shape == STRIPS and route.strip_tiles == 3


# Tiles chosen by the bytes of C that were slower than the larger ones in use before, by up to 1.4 times: deep distances into rows off
# the lines through 128 x 128, and two tiles of 64 rows that read a large image twice.
@pytest.mark.parametrize("dtype, metric, m, n, k, tile", [
    ("e2m3", "euclidean", 78_940, 2733, 12_009, 2), ("i8", "euclidean", 1208, 245_611, 10_624, 2), ("f16", "euclidean", 5825, 48_330, 5312, 2), ("e4m3", "dots", 755, 53_520, 5376, 2),
    ("u4", "euclidean", 90, 251_584, 3306, 3), ("i8", "angular", 79, 269_824, 2122, 3), ("u4", "dots", 74, 178_464, 1664, 3), ("i8", "dots", 216_199, 256, 384, 1)])
def test_larger_tiles_where_the_operands_weigh_most(dtype, metric, m, n, k, tile):
    assert route_of(dtype, metric, m, n, k).shape in (1, 2) if tile < 3 else route_of(dtype, metric, m, n, k).shape == tile


# Three tiles of 64 rows that were taken as four in two of 128, distances of the two-accumulator types (up to 1.4 times the time before).
@pytest.mark.parametrize("dtype, metric, m, n, k", [("e5m2", "angular", 133, 1_285_455, 3780), ("bf16", "euclidean", 133, 419_427, 2376), ("f16", "angular", 192, 252_615, 1731), ("e3m2", "angular", 192, 342_208, 1408)])
def test_rows_of_three_small_tiles(dtype, metric, m, n, k):
    assert route_of(dtype, metric, m, n, k).shape != 3


# Into large C on lines: dots of the two-accumulator types of 3 to 16 stages went through their largest tile, which is slower than it was
# before it folded every two stages, by 1.1 times; 128 x 128 takes two thirds of its time. e2m3 keeps its 128 x 512 tile.
@pytest.mark.parametrize("dtype, m, n, k, shape", [("f16", 4542, 16_384, 324, 3), ("e5m2", 3228, 25_856, 195, 3), ("bf16", 3503, 26_176, 232, 3), ("i4", 4911, 30_208, 288, 3), ("e2m3", 409, 197_504, 960, 5)])
def test_tiles_into_large_results_on_lines(dtype, m, n, k, shape):
    assert route_of(dtype, "dots", m, n, k).shape == shape


# How deep 128 x 128 goes on into rows off the lines (see by_bytes_of_c).
@pytest.mark.parametrize("dtype, metric, m, n, k, shape", [("e4m3", "euclidean", 6080, 40_457, 4682, 3), ("bf16", "dots", 667, 47_635, 5376, 3), ("f16", "euclidean", 5001, 49_001, 5312, 2), ("e2m3", "euclidean", 4000, 40_001, 3500, 1),
                                                           ("u4", "euclidean", 4000, 40_001, 6400, 3)])
def test_depth_of_the_middling_tile(dtype, metric, m, n, k, shape):
    assert route_of(dtype, metric, m, n, k).shape == shape


def _planned(hook, dtype, metric, m, n, k, config=0):
    planned = (ctypes.c_uint32 * 4)()
    nk.library().nk_hip_set_tile_config(config)
    try:
        row = -(-k // DIMENSIONS_PER_VALUE.get(dtype, 1)) * np.dtype(STORAGE[dtype]).itemsize
        assert getattr(nk.library(), hook)(CODES[dtype], {"dots": 0, **METRICS}[metric], m, n, k, 1 << 30, row, 1 << 40, 4 * n, planned) == 0
    finally:
        nk.library().nk_hip_set_tile_config(0)
    return planned[0]


# route_of answers for a call that does not keep A in registers, which is asked first. Of the calls above these do: there what is pinned is
# what they would take without that. All others run as the tests say.
KEEP_A = {("i8", "euclidean", 6718, 20_000, 448), ("u4", "dots", 947, 85_152, 64), ("u4", "dots", 793, 137_216, 317), ("u4", "dots", 161, 1_191_936, 75),
          ("bf16", "dots", 527, 400_384, 192), ("u8", "angular", 1025, 279_648, 1500), ("e4m3", "dots", 407, 580_128, 340),
          ("f16", "dots", 4542, 16_384, 324), ("e5m2", "dots", 3228, 25_856, 195), ("bf16", "dots", 3503, 26_176, 232), ("i4", "dots", 4911, 30_208, 288), ("e2m3", "dots", 409, 197_504, 960)}


@pytest.mark.parametrize("test", [test_no_strips_where_they_do_not_pay, test_strips_where_they_pay, test_short_strips, test_larger_tiles_where_the_operands_weigh_most,
                                  test_rows_of_three_small_tiles, test_tiles_into_large_results_on_lines, test_depth_of_the_middling_tile], ids=lambda test: test.__name__)
def test_which_of_them_keep_a_in_registers(test):
    names = [name.strip() for name in test.pytestmark[0].args[0].split(",")]
    for values in test.pytestmark[0].args[1]:
        call = {"metric": "dots", **dict(zip(names, values))}
        call = tuple(call[name] for name in ("dtype", "metric", "m", "n", "k"))
        assert (_planned("nk_hip_planned_resident", *call) != 0) == (call in KEEP_A), call


# A straight into the LDS of 128 x 128 tiles, on both sides of 257 rows and of 24 stages (of 128 values); not where bit 30 forbids it, nor
# for rows off 16 bytes, u8 (whose bytes are summed on the way), distances.
@pytest.mark.parametrize("dtype, metric, m, k, config, straight", [
    ("i8", "dots", 257, 3072, 3, 1), ("i8", "dots", 256, 3072, 3, 0), ("i8", "dots", 257, 2560, 3, 0), ("i8", "dots", 257, 3200, 3, 0), ("i8", "dots", 257, 3584, 3, 1),
    ("i8", "dots", 4097, 3072, 3 | 1 << 30, 0), ("i8", "dots", 4097, 3500, 3, 0), ("u8", "dots", 4097, 3072, 3, 0), ("i8", "angular", 4097, 3072, 3, 0),
    ("i8", "dots", 2048, 4096, 0, 1), ("i8", "dots", 2048, 2048, 0, 0), ("i8", "dots", 8192, 8192, 0, 1), ("bf16", "dots", 8192, 8192, 0, 1)])
def test_straight_into_lds(dtype, metric, m, k, config, straight):
    assert _planned("nk_hip_planned_direct", dtype, metric, m, max(m, 2048), k, config) == straight
