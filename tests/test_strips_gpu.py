"""Shallow products strip by strip (the part of A of a workgroup stays in LDS, C is written in whole 128-byte lines): the same
bits as through the 64 x 128 tile, and nothing written outside C."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.support import DIMENSIONS_PER_VALUE, STRIPS, route_of
from tests.test_unaligned_gpu import CALLS, DEV, same, values_of

pytestmark = pytest.mark.gpu
STAGE = {"bf16": 64, "f16": 64, "e4m3": 64, "e5m2": 64, "e3m2": 64, "i4": 64, "u4": 64, "u1": 16}  # values stored in a row of one (others: 128)
ALL = ["i8", "u8", "bf16", "f16", "e4m3", "e5m2", "e2m3", "e3m2", "i4", "u4", "u1"]


def through(config, call):
    nk.library().nk_hip_set_tile_config(config)
    try:
        return call()
    finally:
        nk.library().nk_hip_set_tile_config(0)


def framed(m, n, before, after, dtype):
    """C as a window of a larger matrix of one value: rows that start `before` columns into rows of before + n + after."""
    whole = torch.full((m + 2, before + n + after), 77, dtype=dtype, device=DEV)
    return whole, whole[1:m + 1, before:before + n]


def untouched(whole, m, n, before):
    edge = whole.clone()
    edge[1:m + 1, before:before + n] = 77
    return bool((edge == 77).all())


# Rows: a strip of 64 and of 128 rows, one more and less, several. Columns: the fewest, around a tile of 256 and two, a strip that
# ends a few columns into a tile (its last line is all that is left to store) and many strips. Depths: the first two-stage image,
# one value, six stages (the most that 128 rows take), eight and sixteen (64 rows). C: rows on lines, off them by every
# remainder of the row's length, starting off them.
SHAPES = [(33, 128, 2, 0, 0), (64, 129, 2, 3, 1), (65, 255, 4, 0, 1), (127, 256, 6, 0, 0), (128, 257, 6, 31, 9), (129, 513, 5, 1, 2),
          (200, 4104, 1, 5, 0), (300, 5001, 8, 0, 0), (64, 70_003, 16, 2, 3), (513, 20_015, 3, 0, 0), (1000, 33_024, 4, 0, 0)]


@pytest.mark.parametrize("dtype", ALL)
def test_same_bits_as_tiles(dtype):
    rng = np.random.default_rng(81)
    for number, (m, n, stages, before, after) in enumerate(SHAPES):
        columns = stages * STAGE.get(dtype, 128) - (0, 1, 8, 3)[number % 4]
        a, b = values_of(dtype, m, columns, rng).to(DEV), values_of(dtype, min(n, 4099), columns, rng).to(DEV)
        packed = nk.dots_pack(b.repeat(-(-n // 4099), 1)[:n].contiguous(), dtype)
        for metric in ["dots"] if dtype == "u1" else list(CALLS):
            expected = through(4, lambda: CALLS[metric](a, packed))
            whole, window = framed(m, n, before, after, expected.dtype)
            planned = route_of(dtype, metric, m, n, columns * DIMENSIONS_PER_VALUE.get(dtype, 1), STRIPS, 4 * (before + n + after))
            assert planned.shape == STRIPS, f"{dtype} {metric} {m} x {n} x {columns}: not strips, which is what this test is for"
            through(7, lambda: CALLS[metric](a, packed, out=window))
            assert same(window.contiguous(), expected), f"{dtype} {metric} {m} x {n} x {columns}"
            assert untouched(whole, m, n, before), f"{dtype} {metric} {m} x {n} x {columns}: written outside C"


# More pieces of work than there are compute units, so that a workgroup takes a second one (and a third) into the LDS that held the
# first: its rows of A, their sums and norms, what its last lines had left over. (Rows per compute unit, columns, stages, how many
# pieces a workgroup takes at the least): one tile to a piece and two, pieces of 128 rows and of 64, strips beside each other.
@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("rows, n, stages, before, after, least", [(129, 129, 2, 3, 2, 2), (129, 300, 2, 0, 1, 2), (65, 300, 8, 5, 0, 2), (78, 1201, 16, 0, 0, 2), (257, 600, 3, 1, 0, 3)])
def test_workgroups_of_several_pieces(dtype, rows, n, stages, before, after, least):
    units = torch.cuda.get_device_properties(0).multi_processor_count
    m = rows * units
    rng = np.random.default_rng(84)
    columns = stages * STAGE.get(dtype, 128) - 3
    a = values_of(dtype, 4099, columns, rng).to(DEV).repeat(-(-m // 4099), 1)[:m].contiguous() # (4099: no two pieces have the same rows)
    packed = nk.dots_pack(values_of(dtype, n, columns, rng).to(DEV), dtype)
    for metric in ["dots"] if dtype == "u1" else list(CALLS):
        planned = route_of(dtype, metric, m, n, columns * DIMENSIONS_PER_VALUE.get(dtype, 1), STRIPS, 4 * (before + n + after))
        assert planned.shape == STRIPS and planned.units > (least - 1) * units, f"{planned.units} pieces for {units} workgroups"
        expected = through(4, lambda: CALLS[metric](a, packed))
        whole, window = framed(m, n, before, after, expected.dtype)
        through(7, lambda: CALLS[metric](a, packed, out=window))
        assert same(window.contiguous(), expected), f"{dtype} {metric} {m} x {n} x {columns}"
        assert untouched(whole, m, n, before), f"{dtype} {metric} {m} x {n} x {columns}: written outside C"


# NaN and infinities behind the ends of the rows of A (a row of 37 values in rows of 64) stay out of the sums.
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_what_lies_behind_a_row_of_a(dtype):
    rng = np.random.default_rng(82)
    a, b = values_of(dtype, 130, 64, rng).to(DEV), values_of(dtype, 1111, 37, rng).to(DEV)
    expected = through(4, lambda: nk.dots_packed(a[:, :37].contiguous(), nk.dots_pack(b, dtype)))
    a[:, 37:] = float("nan")
    a[::2, 40:] = float("inf")
    assert same(through(7, lambda: nk.dots_packed(a[:, :37], nk.dots_pack(b, dtype))), expected)


# An image of another shape: every result all ones, nothing else written.
@pytest.mark.parametrize("metric", list(CALLS))
def test_image_of_another_product(metric):
    rng = np.random.default_rng(83)
    m, n, k = 70, 3003, 300
    a, b = values_of("i8", m, k, rng).to(DEV), values_of("i8", n, k - 1, rng).to(DEV)
    packed = nk.dots_pack(b, "i8")
    packed.depth = k
    whole, window = framed(m, n, 1, 0, torch.int32 if metric == "dots" else torch.float32)
    try:
        through(7, lambda: CALLS[metric](a, packed, out=window))
    except RuntimeError:
        pass
    assert bool((window.contiguous().view(torch.int32) == -1).all())
    assert untouched(whole, m, n, 1)
