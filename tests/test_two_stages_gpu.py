"""Products of one or two stages of 128 bytes (rows of A of at most 256 bytes, 32 of the bits) take 64 x 128 tiles: the same bits
as through the larger ones, and no slower."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.test_unaligned_gpu import DEV, same, values_of

pytestmark = pytest.mark.gpu
STAGE = {"bf16": 64, "f16": 64, "e4m3": 64, "e5m2": 64, "e3m2": 64, "i4": 64, "u4": 64, "u1": 16}  # values stored in a row of one (others: 128)


def forced(config, call):
    nk.library().nk_hip_set_tile_config(config)
    try:
        return call()
    finally:
        nk.library().nk_hip_set_tile_config(0)


# One stored value, around one stage, at and over two (where the rule ends); rows at the rule's edge and between tiles; a C of
# whole lines, and of 64 KiB from row to row; all pairs, whose tile list follows the shape.
@pytest.mark.parametrize("dtype", ["i8", "u8", "bf16", "f16", "e4m3", "e5m2", "e2m3", "e3m2", "i4", "u4", "u1"])
def test_same_bits_as_the_larger_tiles(dtype):
    rng = np.random.default_rng(71)
    stage = STAGE.get(dtype, 128)
    for m, n, columns in ((127, 16384, stage), (128, 16384, 1), (129, 32768, stage - 1), (257, 8192, 2 * stage), (1000, 4128, stage + 1), (300, 8192, 2 * stage + 1)):
        a, b = values_of(dtype, m, columns, rng).to(DEV), values_of(dtype, n, columns, rng).to(DEV)
        packed = nk.dots_pack(b, dtype)
        assert same(nk.dots_packed(a, packed), forced(3, lambda: nk.dots_packed(a, packed))), f"{dtype} {m} x {n} x {columns}"
    for count in (1500, 2500):
        vectors = values_of(dtype, count, 2 * stage, rng).to(DEV)
        assert same(nk.dots_symmetric(vectors, dtype), forced(3, lambda: nk.dots_symmetric(vectors, dtype))), f"{dtype} all pairs of {count}"


# (The 128 x 256 tile once took 1.24 times as long as 128 x 128 here. Best of five in turn; runs of one side differ by 2 per cent.)
@pytest.mark.parametrize("dtype", ["e4m3", "e5m2"])
def test_no_slower_than_a_middling_tile(dtype):
    rng = np.random.default_rng(72)
    m, n, k = 2000, 262_144, 128
    packed = nk.dots_pack(values_of(dtype, 4096, k, rng).to(DEV).repeat(n // 4096, 1), dtype)
    a, out = values_of(dtype, m, k, rng).to(DEV), torch.empty((m, n), dtype=torch.float32, device=DEV)
    best = {}
    for _ in range(5):
        for config in (0, 3):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(4):
                forced(config, lambda: nk.dots_packed(a, packed, out=out))
            end.record()
            end.synchronize()
            best[config] = min(best.get(config, 1e9), begin.elapsed_time(end) / 4)
    assert best[0] <= 1.12 * best[3], f"{dtype}: {best[0]:.3f} ms chosen, {best[3]:.3f} ms through 128 x 128"
