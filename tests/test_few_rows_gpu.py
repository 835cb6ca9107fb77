"""Products of few rows, and of few tiles, run through a tile of 32 rows: the same bits as through the 64-row tile."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.test_unaligned_gpu import CALLS, DEV, placed, same, values_of

pytestmark = pytest.mark.gpu


# Rows around the tile's 32 and the next tile's 64; columns around one and several tiles of 128; rows of A under four
# stages of 128 bytes (no pipeline across tiles), at them, of whole stages and not, and at odd addresses.
@pytest.mark.parametrize("dtype", ["i8", "u8", "bf16", "f16", "e4m3", "e5m2", "e2m3", "e3m2", "i4", "u4", "u1"])
def test_few_rows_give_the_bits_of_the_larger_tile(dtype):
    rng = np.random.default_rng(41)
    for m, n, cols in ((1, 1, 1), (1, 129, 300), (31, 257, 512), (32, 128, 1024), (33, 33, 513), (64, 300, 520), (95, 1000, 1100)):
        a, b = values_of(dtype, m, cols, rng), values_of(dtype, n, cols, rng)
        packed = nk.dots_pack(b.to(DEV), dtype)
        for offset in (0, 1):
            rows = placed(a, offset, offset)
            for metric in ["dots"] if dtype == "u1" else list(CALLS):
                results = {}
                for config in (4, 6, 0):
                    nk.library().nk_hip_set_tile_config(config)
                    try:
                        results[config] = CALLS[metric](rows, packed)
                    finally:
                        nk.library().nk_hip_set_tile_config(0)
                assert same(results[6], results[4]), f"{dtype} {metric} {m}x{n}x{cols} offset {offset}"
                assert same(results[0], results[4]), f"{dtype} {metric} {m}x{n}x{cols} offset {offset}, tile chosen by the library"


# Many tiles for every workgroup (2344 tiles of 32 x 128, at most 1024 workgroups of them at once). The table is one of 4099
# vectors over and over, so every stretch of 4099 columns must hold the bits that a product of those alone gives: 33 tiles,
# one to a workgroup. Depths of five stages of 128 bytes (16 for the bits), dword-aligned rows and odd ones.
@pytest.mark.parametrize("dtype", ["i8", "u8", "bf16", "f16", "e4m3", "e5m2", "e2m3", "e3m2", "i4", "u4", "u1"])
def test_few_rows_across_tiles(dtype):
    rng = np.random.default_rng(42)
    n, distinct = 300_003, 4099
    columns = {"bf16": 300, "f16": 300, "i4": 300, "u4": 300, "e4m3": 300, "e5m2": 300, "e3m2": 300, "u1": 76}.get(dtype, 600)
    b = values_of(dtype, distinct, columns, rng).to(DEV)
    times = -(-n // distinct)
    packed, alone = nk.dots_pack(b.repeat(times, 1)[:n].contiguous(), dtype), nk.dots_pack(b, dtype)
    for m in (1, 31, 32):
        a = values_of(dtype, m, columns, rng)
        for offset in (0, 1):
            rows = placed(a, offset, offset)
            for metric in ["dots"] if dtype == "u1" else list(CALLS):
                got, once = CALLS[metric](rows, packed), CALLS[metric](rows, alone)
                assert same(got, once.repeat(1, times)[:, :n].contiguous()), f"{dtype} {metric} {m} rows offset {offset}"
                del got
