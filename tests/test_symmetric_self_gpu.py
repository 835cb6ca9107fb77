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
        if count > 64: # windows on a tile of the image (A out of it, its sums too) and off it (A and its sums from the vectors)
            for metric in ["dots"] if dtype == "u1" else list(CALLS):
                whole = SYMMETRIC[metric](vectors, dtype).view(torch.int32)
                for start in (32, 45):
                    part = SYMMETRIC[metric](vectors, dtype, start_row=start, end_row=count - 3).view(torch.int32)
                    assert torch.equal(torch.triu(part)[start:count - 3], torch.triu(whole)[start:count - 3]), f"{dtype} {metric} rows {start} on of {count} x {columns}"


# Values of many magnitudes, whose squares span more than f64 can add without rounding. The packing launch adds a row's squares in another
# order than the loop does; the two are within 2^-42 of each other (600 additions in f64 each), so that rounded to f32 they can
# differ for one row in 2^18 at the most. These rows do not.
@pytest.mark.parametrize("dtype, spread", [("bf16", 9.0), ("f16", 3.0)])
def test_row_sums_of_many_magnitudes(dtype, spread):
    rng = np.random.default_rng(92)
    count, columns = 700, 600
    values = rng.standard_normal((count, columns)) * 10.0 ** rng.uniform(-spread, spread, (count, columns))
    vectors = torch.from_numpy(values.astype(np.float32)).to(torch.bfloat16 if dtype == "bf16" else torch.float16).to(DEV)
    assert not bool(torch.isinf(vectors).any())
    packed = nk.dots_pack(vectors, dtype)
    for metric in ("angular", "euclidean"):
        full = torch.triu(CALLS[metric](vectors, packed).view(torch.int32), 1)
        assert torch.equal(torch.triu(SYMMETRIC[metric](vectors, dtype).view(torch.int32)), full), f"{dtype} {metric}"
        for start in (32, 45):
            part = SYMMETRIC[metric](vectors, dtype, start_row=start, end_row=count).view(torch.int32)
            assert torch.equal(torch.triu(part)[start:], full[start:]), f"{dtype} {metric} rows {start} on"
