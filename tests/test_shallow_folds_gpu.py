"""Folds of shallow products of the two-accumulator types: after every trip of the loop, the same bits as where they are counted."""
import numpy as np
import pytest

import numkong_amd as nk
from tests.test_unaligned_gpu import CALLS, DEV, same, values_of

pytestmark = pytest.mark.gpu
STAGE = 64  # values stored in a row of one stage


def through(config, call):
    nk.library().nk_hip_set_tile_config(config)
    try:
        return call()
    finally:
        nk.library().nk_hip_set_tile_config(0)


# Folds: the two-accumulator types through tiles that fold after every trip of the loop (up to 31 stages) and the 32 x 128 tile,
# which looks every time whether a fold is due; 4, 6, 30 and 31 stages, and 32, where folds become rarer.
@pytest.mark.parametrize("dtype", ["bf16", "f16", "e4m3", "e5m2", "e3m2"])
def test_folds_of_shallow_products(dtype):
    rng = np.random.default_rng(84)
    for stages, less in ((4, 0), (4, 1), (6, 2), (30, 0), (30, 1), (31, 8), (32, 0)):
        columns = stages * STAGE - less
        a, b = values_of(dtype, 257, columns, rng).to(DEV), values_of(dtype, 515, columns, rng).to(DEV)
        packed = nk.dots_pack(b, dtype)
        for metric in CALLS:
            expected = through(6, lambda: CALLS[metric](a, packed))
            for config in (2, 3, 4):
                assert same(through(config, lambda: CALLS[metric](a, packed)), expected), f"{dtype} {metric} {columns} through shape {config}"
