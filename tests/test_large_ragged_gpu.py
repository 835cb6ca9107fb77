"""Results larger than the last-level cache with rows off the 128-byte lines: the same bits as through the 64-row tile."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.test_unaligned_gpu import DEV, same, values_of

pytestmark = pytest.mark.gpu


# One shape for each tile that the rule picks by depth (in stages of 128 bytes of operand), its rows not a multiple of any
# tile, and the smallest C that the rule takes for large.
@pytest.mark.parametrize("dtype", ["i8", "u8", "i4", "u1", "e2m3", "bf16", "f16", "e4m3"])
def test_tiles_of_large_results(dtype):
    rng = np.random.default_rng(61)
    values = {"bf16": 64, "f16": 64, "e4m3": 64, "i4": 64, "u1": 16}.get(dtype, 128)  # stored in a row of a stage
    for m, n, stages in ((133, 760_003, 2), (133, 760_003, 4), (129, 790_001, 6), (257, 393_003, 10), (300, 120_001, 18)):
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
