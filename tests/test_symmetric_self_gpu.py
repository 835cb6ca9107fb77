"""All pairs with A out of the packed image: the same bits as where A is staged from the vectors (a window that does not start on
a tile of the image), and as the packed kinds with both sides the same."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.test_unaligned_gpu import CALLS, DEV, values_of

pytestmark = pytest.mark.gpu
STAGE = {"bf16": 64, "f16": 64, "e4m3": 64, "e5m2": 64, "e3m2": 64, "i4": 64, "u4": 64, "u1": 16}  # values stored in a row of one (others: 128)
SYMMETRIC = {"dots": nk.dots_symmetric, "angular": nk.angulars_symmetric, "euclidean": nk.euclideans_symmetric}


# Vectors: around a tile of the image, several tile rows, several bands of 8 of them with a last band that is short. Depths: four
# stages (the pipeline's least), five (an image of six), around the 32 where folds become rarer, odd numbers of bytes.
@pytest.mark.parametrize("dtype", ["i8", "u8", "bf16", "f16", "e4m3", "e5m2", "e2m3", "e3m2", "i4", "u4", "u1"])
def test_same_bits_as_both_sides_packed(dtype):
    rng = np.random.default_rng(91)
    stage = STAGE.get(dtype, 128)
    for count, columns in ((1, 4 * stage), (33, 4 * stage - 1), (257, 5 * stage), (700, 31 * stage + 1), (1100, 3 * stage + 1), (2100, 33 * stage)):
        vectors = values_of(dtype, count, columns, rng).to(DEV)
        packed = nk.dots_pack(vectors, dtype)
        for metric in ["dots"] if dtype == "u1" else list(CALLS):
            full = CALLS[metric](vectors, packed).view(torch.int32)
            full = torch.triu(full, 1 if metric != "dots" else 0) # (a vector's distance from itself is 0 in the symmetric kinds)
            for config in (0, 2, 3, 4):
                nk.library().nk_hip_set_tile_config(config)
                try:
                    got = SYMMETRIC[metric](vectors, dtype).view(torch.int32)
                finally:
                    nk.library().nk_hip_set_tile_config(0)
                assert torch.equal(torch.triu(got), full), f"{dtype} {metric} {count} x {columns} shape {config}"
        if count > 64: # windows on a tile of the image and off it
            whole = SYMMETRIC["dots"](vectors, dtype)
            for start in (32, 45):
                part = SYMMETRIC["dots"](vectors, dtype, start_row=start, end_row=count - 3)
                assert torch.equal(torch.triu(part)[start:count - 3], torch.triu(whole)[start:count - 3]), f"{dtype} rows {start} on of {count} x {columns}"
