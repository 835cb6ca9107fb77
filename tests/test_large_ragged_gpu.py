"""Results larger than the last-level cache with rows off the 128-byte lines: the same bits as through the 64-row tile."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.test_unaligned_gpu import DEV, same, values_of

pytestmark = pytest.mark.gpu


# One shape for each tile that the rule picks by depth (in stages of 128 bytes of operand), its rows not a multiple of any
# tile, and the smallest C that the rule takes for large; 300 rows at six stages are an odd number of 128s, where the
# integers leave the 256-row tile. (e2m3 takes its 128 x 512 tile for all of these: there are 256 of them each time. It is
# here for that tile's masked stores into such rows.)
@pytest.mark.parametrize("dtype", ["i8", "u8", "i4", "u1", "e2m3", "bf16", "f16", "e4m3"])
def test_tiles_of_large_results(dtype):
    rng = np.random.default_rng(61)
    values = {"bf16": 64, "f16": 64, "e4m3": 64, "i4": 64, "u1": 16}.get(dtype, 128)  # stored in a row of a stage
    for m, n, stages in ((133, 760_003, 2), (133, 760_003, 4), (129, 790_001, 6), (300, 340_003, 6), (257, 393_003, 10), (300, 120_001, 18)):
        columns = stages * values - 8 * (values > 16)
        a, b = values_of(dtype, m, columns, rng).to(DEV), values_of(dtype, 4099, columns, rng)
        packed = nk.dots_pack(b.to(DEV).repeat(-(-n // 4099), 1)[:n].contiguous(), dtype)
        chosen = nk.dots_packed(a, packed)
        nk.library().nk_hip_set_tile_config(4)
        try:
            expected = nk.dots_packed(a, packed)
        finally:
            nk.library().nk_hip_set_tile_config(0)
        assert same(chosen, expected), f"{dtype} {m} x {n} x {columns}"
        del packed, chosen, expected


# Shapes that a rule for such results once made slower than the tile it replaced (by 1.22 to 1.44 times): whatever is chosen now
# may not take more than 1.12 times as long as that tile. (Runs of one side differ by 2 per cent at most, best of five, in turn.)
@pytest.mark.parametrize("dtype, m, n, k, tile", [("i8", 1000, 209_697, 1700, 1), ("i8", 512, 409_601, 1700, 1), ("u8", 512, 409_601, 1700, 1),
                                                  ("i8", 2400, 45_872, 400, 4), ("u8", 2400, 45_872, 400, 4), ("bf16", 2400, 45_872, 900, 4)])
def test_no_slower_than_the_tile_of_smaller_results(dtype, m, n, k, tile):
    rng = np.random.default_rng(62)
    a, b = values_of(dtype, m, k, rng).to(DEV), values_of(dtype, 4099, k, rng).to(DEV)
    packed = nk.dots_pack(b.repeat(-(-n // 4099), 1)[:n].contiguous(), dtype)
    out = torch.empty((m, n), dtype=torch.float32 if dtype == "bf16" else torch.int32, device=DEV)
    best = {}
    for _ in range(5):
        for config in (0, tile):
            nk.library().nk_hip_set_tile_config(config)
            try:
                begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                begin.record()
                for _ in range(4):
                    nk.dots_packed(a, packed, out=out)
                end.record()
                end.synchronize()
            finally:
                nk.library().nk_hip_set_tile_config(0)
            best[config] = min(best.get(config, 1e9), begin.elapsed_time(end) / 4)
    assert best[0] <= 1.12 * best[tile], f"{dtype} {m} x {n} x {k}: {best[0]:.3f} ms chosen, {best[tile]:.3f} ms through shape {tile}"


# Partial lines of many rows past the caches: two workgroups on a compute unit took 1.2 and 1.15 times as long as one of the 128 x 256 tile
# does (one of 128 x 128: 1.03 and 0.91). Results are new ones in turn: into one that the last-level cache holds all are alike.
@pytest.mark.parametrize("dtype, m, n, k, tile", [("bf16", 1_000_000, 130, 768, 2), ("bf16", 1_536_789, 218, 382, 2)])
def test_rows_past_the_caches(dtype, m, n, k, tile):
    rng = np.random.default_rng(63)
    a = values_of(dtype, 4099, k, rng).to(DEV).repeat(-(-m // 4099), 1)[:m].contiguous()
    packed = nk.dots_pack(values_of(dtype, n, k, rng).to(DEV), dtype)
    outs = [torch.empty((m, n), dtype=torch.float32, device=DEV) for _ in range(3)]
    best = {}
    for _ in range(5):
        for config in (0, tile):
            nk.library().nk_hip_set_tile_config(config)
            try:
                begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                begin.record()
                for out in outs:
                    nk.dots_packed(a, packed, out=out)
                end.record()
                end.synchronize()
            finally:
                nk.library().nk_hip_set_tile_config(0)
            best[config] = min(best.get(config, 1e9), begin.elapsed_time(end) / 3)
    assert best[0] <= 1.1 * best[tile], f"{dtype} {m} x {n} x {k}: {best[0]:.3f} ms chosen, {best[tile]:.3f} ms through shape {tile}"
