"""Rows of A and B at any byte address: the shifted loads of the product and of the pack kernel (an odd depth of bytes, an
odd depth of 16-bit values, matrices that start off a dword), on a real MI355X.

Where the bytes lie must not change a bit of the result: the same operands in aligned memory, which the other tests hold
to the oracle, give the expected values, for every element type that is not f32 or f64, every tile shape and metric.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import numkong_amd as nk  # noqa: E402
from numkong_amd import api  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NARROWER = [d for d in api.DTYPES if d not in ("f32", "f64")]
CALLS = {"dots": nk.dots_packed, "angular": nk.angulars_packed, "euclidean": nk.euclideans_packed}


def values_of(dtype, rows, cols, rng):
    """Stored values of every kind the type has, as bytes or 16-bit words; no infinities or NaNs, which compare unequal."""
    if dtype in ("bf16", "f16"):
        return torch.from_numpy(rng.standard_normal((rows, cols)).astype(np.float32)).to(torch.bfloat16 if dtype == "bf16" else torch.float16)
    raw = rng.integers(0, 256, size=(rows, cols), dtype=np.uint8)
    if dtype in ("e4m3", "e5m2"):
        raw = np.where((raw & 0x7F) > 0x7B, raw & 0xF0, raw) & (0x9F if dtype == "e5m2" else 0xFF)
    return torch.from_numpy(raw.view(np.int8) if dtype == "i8" else raw)


def placed(values, pad, offset):
    """The same values on the GPU, `offset` values into rows that are `pad` values longer. What lies around them is NaN in
    the float types (0x7F is one of both fp8 types): times the zeros that an image's depth is padded with, anything else
    would vanish, whether or not the kernel masks what it reads past a row's end."""
    rows, cols = values.shape
    around = float("nan") if values.dtype.is_floating_point else 0x7F
    whole = torch.full((rows, cols + pad + offset), around, dtype=values.dtype).to(DEV)
    view = whole[:, offset:offset + cols]
    view.copy_(values)
    return view


def aligned(values):
    per = 16 // values.element_size()
    return placed(values, (-values.shape[1]) % per, 0)


def same(got, expected):
    return torch.equal(got.view(torch.int32), expected.view(torch.int32))


# Stored values per row: just under, at and over a whole number of 128-byte stages (even and odd numbers of them), four
# stages at least, and one row of a single value past it.
@pytest.mark.parametrize("dtype", NARROWER)
@pytest.mark.parametrize("config", [0, 1, 2, 3, 4])
def test_unaligned_rows_give_the_aligned_bits(dtype, config):
    rng = np.random.default_rng(31 + config)
    width = api.DTYPES[dtype][1]
    for m, n, row_bytes in ((1, 33, 513), (67, 130, 767), (130, 257, 1025), (257, 300, 1279)):
        cols = row_bytes if width == 1 else (row_bytes // 2) | 1
        if dtype == "u1":
            cols = cols // 8 + 60 | 1  # four stages of 16 bytes at least
        a, b = values_of(dtype, m, cols, rng), values_of(dtype, n, cols, rng)
        packed = nk.dots_pack(aligned(b), dtype)
        metrics = ["dots"] if dtype == "u1" else list(CALLS)
        nk.library().nk_hip_set_tile_config(config)
        try:
            expected = {metric: CALLS[metric](aligned(a), packed) for metric in metrics}
            for pad, offset in ((0, 0), (2, 1), (0, 2), (1, 3)):
                for metric in metrics:
                    got = CALLS[metric](placed(a, pad, offset), packed)
                    assert same(got, expected[metric]), f"{dtype} {metric} {m}x{n}x{cols} pad {pad} offset {offset}"
        finally:
            nk.library().nk_hip_set_tile_config(0)


# Many tiles for every workgroup (the largest device-resident grid is 1024 workgroups; the fewest tiles here are 2193 of
# 128 x 256): what a tile's last stages fetch is the next tile's first stages, shifted as its base asks, and the sums that
# the staging keeps (u8's rows, the distances' squares) change sets with every tile.
@pytest.mark.parametrize("dtype", NARROWER)
@pytest.mark.parametrize("config", [0, 2, 3, 4, 6])
def test_unaligned_rows_across_tiles(dtype, config):
    rng = np.random.default_rng(33)
    m, n = 2100, 33_001
    cols = 125 if dtype == "u1" else 515
    a, b = values_of(dtype, m, cols, rng), values_of(dtype, 4099, cols, rng)
    packed = nk.dots_pack(b.to(DEV).repeat(-(-n // 4099), 1)[:n].contiguous(), dtype)
    for metric in ["dots"] if dtype == "u1" else list(CALLS):
        nk.library().nk_hip_set_tile_config(config)
        try:
            expected = CALLS[metric](aligned(a), packed)
            for pad, offset in ((0, 0), (1, 1)):
                got = CALLS[metric](placed(a, pad, offset), packed)
                assert same(got, expected), f"{dtype} {metric} config {config} pad {pad} offset {offset}"
        finally:
            nk.library().nk_hip_set_tile_config(0)


# Rows of one or two stages, where the pipeline starts anew with every tile: one byte, under, at and over one stage of 128
# bytes (16 of the bits), the last odd length before four stages; one tile, and many for every workgroup.
@pytest.mark.parametrize("dtype", NARROWER)
@pytest.mark.parametrize("config", [0, 1, 2, 3, 4, 6])
def test_unaligned_rows_of_two_stages(dtype, config):
    rng = np.random.default_rng(34)
    width = api.DTYPES[dtype][1]
    stage = {"u1": 16, "i4": 64, "u4": 64, "e4m3": 64, "e5m2": 64, "e3m2": 64}.get(dtype, 128 // width)  # values stored in a row of one
    for m, n, cols in ((1, 1, 1), (33, 70, 5), (67, 130, stage - 1), (130, 257, stage), (257, 300, stage + 1), (2100, 33_001, 2 * stage - 1)):
        a, b = values_of(dtype, m, cols, rng), values_of(dtype, min(n, 4099), cols, rng)
        packed = nk.dots_pack(b.to(DEV).repeat(-(-n // 4099), 1)[:n].contiguous(), dtype)
        nk.library().nk_hip_set_tile_config(config)
        try:
            for metric in ["dots"] if dtype == "u1" else list(CALLS):
                expected = CALLS[metric](aligned(a), packed)
                for pad, offset in ((0, 0), (0, 1), (2, 1), (1, 3)):
                    got = CALLS[metric](placed(a, pad, offset), packed)
                    assert same(got, expected), f"{dtype} {metric} {m}x{n}x{cols} config {config} pad {pad} offset {offset}"
        finally:
            nk.library().nk_hip_set_tile_config(0)


@pytest.mark.parametrize("dtype", NARROWER)
def test_unaligned_rows_pack_to_the_aligned_image(dtype):
    rng = np.random.default_rng(32)
    for n, cols in ((1, 1), (33, 17), (70, 301), (40, 1025)):
        b = values_of(dtype, n, cols, rng)
        expected = nk.dots_pack(aligned(b), dtype).buffer.clone()
        for pad, offset in ((0, 0), (2, 1), (0, 2), (1, 3)):
            got = nk.dots_pack(placed(b, pad, offset), dtype).buffer.clone()
            for image in (got, expected):
                image[32:40] = 0  # (the number of the pack call)
            assert torch.equal(got, expected), f"{dtype} {n}x{cols} pad {pad} offset {offset}"
