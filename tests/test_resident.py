"""Shallow products with A in registers: which calls take them, the same bits as through the 64 x 128 tile, nothing written outside C."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.support import CODES, DIMENSIONS_PER_VALUE, METRICS, STORAGE
from tests.test_strips_gpu import STAGE, framed, through, untouched
from tests.test_unaligned_gpu import CALLS, DEV, aligned, placed, same, values_of

TYPES = ["i8", "u8", "bf16", "f16", "e4m3", "e5m2", "e2m3", "e3m2", "i4", "u4"]
FLOATS = ["bf16", "f16", "e4m3", "e5m2", "e3m2"]


def resident_of(dtype, metric, m, n, k, config=0, row_bytes=0):
    """(rows of a wavefront, workgroups, tiles of a strip) of a call that keeps A in registers, (0, 0, 0) of any other."""
    planned = (ctypes.c_uint32 * 3)()
    a_row = -(-k // DIMENSIONS_PER_VALUE.get(dtype, 1)) * np.dtype(STORAGE[dtype]).itemsize
    nk.library().nk_hip_set_tile_config(config)
    try:
        status = nk.library().nk_hip_planned_resident(CODES[dtype], {"dots": 0, **METRICS}[metric], m, n, k, 1 << 30, a_row, 1 << 40, row_bytes or 4 * n, planned)
    finally:
        nk.library().nk_hip_set_tile_config(0)
    assert status == 0, nk.library().nk_hip_last_error()
    return tuple(planned)


def built(dtype, metric, stages, blocks, lines):
    """Is there a kernel for the stages of an image (an even number), one block of 32 rows per wavefront or two?"""
    floats = dtype in FLOATS
    if blocks == 2:
        return metric == "dots" and lines and stages <= (4 if floats else 6)
    if metric == "angular" and (stages > 8 if floats else stages < 4):
        return False
    return stages <= (10 if floats else 12) if lines else (8 if metric == "angular" else 6) <= stages <= 10 and not (metric == "angular" and floats and stages > 8)


def test_calls_that_keep_a_in_registers():
    assert resident_of("i8", "dots", 1024, 1_048_576, 768)[0] == 64 and resident_of("i8", "dots", 1000, 500_032, 300)[0] == 64
    assert resident_of("f16", "dots", 8192, 8191, 500)[0] == 32 and resident_of("i8", "angular", 1024, 524_288, 768)[0] == 32
    for dtype, metric, m, n, k in [("i8", "dots", 64, 1_048_576, 768), ("i8", "dots", 8192, 8192, 8192), ("u8", "euclidean", 1000, 500_009, 301), ("f16", "dots", 8192, 8191, 1000),
                                   ("u1", "dots", 1024, 1_048_576, 768), ("i8", "dots", 1000, 10_000, 768), ("f16", "angular", 128, 1_000_000, 500), ("i8", "dots", 100_000, 352, 768)]:
        assert resident_of(dtype, metric, m, n, k) == (0, 0, 0), (dtype, metric, m, n, k)


def test_which_kernels_there_are():
    for dtype in TYPES + ["u1"]:
        for metric in ["dots"] if dtype == "u1" else ["dots", *METRICS]:
            for stages in range(2, 18, 2):
                for blocks in (1, 2):
                    for n in (1024, 1025):
                        k = stages * STAGE.get(dtype, 128) * DIMENSIONS_PER_VALUE.get(dtype, 1)
                        rows = resident_of(dtype, metric, 100, n, k, 7 + blocks)[0]
                        assert rows == (32 * blocks if dtype != "u1" and built(dtype, metric, stages, blocks, n == 1024) else 0), (dtype, metric, stages, blocks, n)


# Rows: one, around a block of 32, two wavefronts and all eight, workgroups that share them out unevenly. Columns: one, around a tile of
# 32, fewer tiles than the ring holds and a few more, a strip that ends a few columns into a tile (off the lines the rest of its last
# line is all that is left to store), several strips. Depths: every number of stages, whole and short of it by one value and by
# more than a stage. C: rows on lines, off them by every remainder of the row's length, starting off them.
SHAPES = [(1, 1, 2, 0, 31), (31, 33, 4, 0, 31), (32, 64, 6, 0, 0), (33, 95, 8, 0, 1), (64, 127, 10, 1, 0), (65, 4099, 6, 0, 0), (255, 160, 12, 0, 0), (257, 8197, 8, 3, 4),
          (520, 1057, 10, 31, 2), (300, 12_000, 4, 0, 0), (700, 9001, 6, 0, 23), (1000, 40_003, 2, 0, 29), (129, 5, 8, 2, 1), (600, 3333, 12, 0, 27)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", TYPES)
def test_same_bits_as_tiles(dtype):
    rng = np.random.default_rng(91)
    ran = 0
    for number, (m, n, stages, before, after) in enumerate(SHAPES):
        columns = stages * STAGE.get(dtype, 128) - (0, 1, 8, STAGE.get(dtype, 128) + 3)[number % 4]
        # (every other A starts on an odd element of rows of an odd length)
        wide, odd = values_of(dtype, m, columns + 3, rng).to(DEV), number % 2
        a = wide[:, odd:columns + odd] if odd else wide[:, :columns].contiguous()
        packed = nk.dots_pack(values_of(dtype, min(n, 4099), columns, rng).to(DEV).repeat(-(-n // 4099), 1)[:n].contiguous(), dtype)
        k, lines = columns * DIMENSIONS_PER_VALUE.get(dtype, 1), (before + n + after) % 32 == 0 and before == 0
        for metric in CALLS:
            for blocks in (1, 2):
                if not built(dtype, metric, stages, blocks, lines):
                    continue
                expected = through(4, lambda: CALLS[metric](a, packed))
                whole, window = framed(m, n, before, after, expected.dtype)
                through(7 + blocks, lambda: CALLS[metric](a, packed, out=window))
                assert same(window.contiguous(), expected), f"{dtype} {metric} {m} x {n} x {columns}, {blocks} blocks"
                assert untouched(whole, m, n, before), f"{dtype} {metric} {m} x {n} x {columns}, {blocks} blocks: written outside C"
                ran += 1
    assert ran >= 12


# More pieces of work than compute units, chosen without being asked for, and rows of A that repeat themselves (stride 0).
@pytest.mark.gpu
@pytest.mark.parametrize("dtype, metric, m, n, k", [("i8", "dots", 120_001, 1088, 500), ("bf16", "euclidean", 60_000, 544, 300), ("u8", "angular", 400, 70_016, 900), ("e4m3", "dots", 4000, 8705, 500)])
def test_chosen(dtype, metric, m, n, k):
    rng = np.random.default_rng(92)
    a = values_of(dtype, 4099, k, rng).to(DEV).repeat(-(-m // 4099), 1)[:m].contiguous()
    packed = nk.dots_pack(values_of(dtype, min(n, 4099), k, rng).to(DEV).repeat(-(-n // 4099), 1)[:n].contiguous(), dtype)
    assert resident_of(dtype, metric, m, n, k)[0]
    assert same(CALLS[metric](a, packed), through(4, lambda: CALLS[metric](a, packed)))
    flat = a[:1].expand(m, k)
    assert same(CALLS[metric](flat, packed), through(4, lambda: CALLS[metric](flat.contiguous(), packed)))


# NaN and infinities behind the ends of the rows of A stay out of the sums, on lines and off them.
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("n", [1024, 1111])
def test_what_lies_behind_a_row_of_a(dtype, n):
    rng = np.random.default_rng(93)
    a, b = values_of(dtype, 130, 500, rng).to(DEV), values_of(dtype, n, 421, rng).to(DEV)
    expected = through(4, lambda: nk.dots_packed(a[:, :421].contiguous(), nk.dots_pack(b, dtype)))
    a[:, 421:] = float("nan")
    a[::2, 424:] = float("inf")
    assert resident_of(dtype, "dots", 130, n, 421, 8)[0] == 32
    assert same(through(8, lambda: nk.dots_packed(a[:, :421], nk.dots_pack(b, dtype))), expected)


# An image of another shape: every result all ones, nothing else written.
@pytest.mark.gpu
@pytest.mark.parametrize("metric", list(CALLS))
@pytest.mark.parametrize("n, before", [(3003, 1), (3008, 0)])
def test_image_of_another_product(metric, n, before):
    rng = np.random.default_rng(94)
    m, k = 300, 1000
    a, b = values_of("i8", m, k, rng).to(DEV), values_of("i8", n, k - 1, rng).to(DEV)
    packed = nk.dots_pack(b, "i8")
    packed.depth = k
    whole, window = framed(m, n, before, 0, torch.int32 if metric == "dots" else torch.float32)
    assert resident_of("i8", metric, m, n, k, 8, 4 * (before + n))[0] == 32
    try:
        through(8, lambda: CALLS[metric](a, packed, out=window))
    except RuntimeError:
        pass
    assert bool((window.contiguous().view(torch.int32) == -1).all())
    assert untouched(whole, m, n, before)


# Nothing in the loop over the tiles is reloaded from memory: such a load would wait for all stores in front of it. (One register may be
# saved around the loading of A; u4 angular of ten stages off the lines spilled 16, and took 1.05 of the time of the tiles it replaces.)
def test_registers_hold_a(tmp_path):
    tools = "/opt/rocm/llvm/bin"
    if not os.path.exists(f"{tools}/llvm-objdump"):
        pytest.skip("no llvm-objdump")
    library = shutil.copy(nk.api.library_path(), tmp_path)
    subprocess.run([f"{tools}/llvm-objdump", "--offloading", library], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    spilled, kernels = {}, 0
    for part in tmp_path.glob("*gfx950"):
        name = None
        for line in subprocess.run([f"{tools}/llvm-readelf", "--notes", part], check=True, capture_output=True, text=True).stdout.splitlines():
            if line.strip().startswith(".name:"):
                name = line.split()[-1]
            elif ".vgpr_spill_count:" in line and "dots_resident_kernel" in name:
                kernels += 1
                if int(line.split()[-1]) > 1:
                    spilled[name] = int(line.split()[-1])
    assert kernels > 150 and not spilled


# The deeper kernels on lines, whose rings of LDS differ (four tiles at eight stages, three at ten and twelve): more rows than a workgroup
# has, several strips, each longer than the ring, a strip that ends nine columns into a tile; depths whole, short by one, by eight values
# and by more than a stage.
@pytest.mark.gpu
@pytest.mark.parametrize("stages", [8, 10, 12])
@pytest.mark.parametrize("dtype", TYPES)
def test_deeper_on_lines(dtype, stages):
    rng = np.random.default_rng(96)
    m, ran = 777, 0
    for n, after, short in ((20_000, 0, 0), (19_977, 23, 1), (20_000, 32, 8), (19_977, 23, STAGE.get(dtype, 128) + 3)):
        columns = stages * STAGE.get(dtype, 128) - short
        a = values_of(dtype, m, columns, rng).to(DEV)
        packed = nk.dots_pack(values_of(dtype, 4099, columns, rng).to(DEV).repeat(5, 1)[:n].contiguous(), dtype)
        for metric in CALLS:
            if not built(dtype, metric, stages, 1, True):
                continue
            rows, units, tiles = resident_of(dtype, metric, m, n, columns * DIMENSIONS_PER_VALUE.get(dtype, 1), 8, 4 * (n + after))
            assert rows == 32 and units >= 40 and tiles > 4, f"{units} pieces of {tiles} tiles"
            expected = through(4, lambda: CALLS[metric](a, packed))
            whole, window = framed(m, n, 0, after, expected.dtype)
            through(8, lambda: CALLS[metric](a, packed, out=window))
            assert same(window.contiguous(), expected), f"{dtype} {metric} {m} x {n} x {columns}"
            assert untouched(whole, m, n, 0), f"{dtype} {metric} {m} x {n} x {columns}: written outside C"
            ran += 1
    assert ran >= 4 or (dtype in FLOATS and stages == 12)


# NaN around the rows of A for the types whose chunks are 8 bytes as well, rows that start on odd addresses, an image of which almost two
# stages are empty: seven hold values, the seventh a single one.
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "f16", "e4m3", "e5m2"])
@pytest.mark.parametrize("metric", list(CALLS))
@pytest.mark.parametrize("n", [1024, 1111])
def test_nan_around_the_rows_of_a(dtype, metric, n):
    rng = np.random.default_rng(97)
    a, b = values_of(dtype, 300, 385, rng), values_of(dtype, n, 385, rng)
    packed = nk.dots_pack(aligned(b), dtype)
    expected = through(4, lambda: CALLS[metric](aligned(a), packed))
    assert resident_of(dtype, metric, 300, n, 385, 8)[0] == 32
    for pad, offset in ((131, 0), (130, 1), (128, 3), (64, 1)):
        assert same(through(8, lambda: CALLS[metric](placed(a, pad, offset), packed)), expected), f"{pad} values behind, {offset} in front"


# Both sides of the lines of the rule: rows, bytes of C, tiles of a strip, wavefronts with rows (angular), floats of eight stages off the lines
# with few rows, two blocks of rows by image and rows.
@pytest.mark.parametrize("dtype, metric, m, n, k, rows", [
    ("i8", "dots", 64, 1_048_576, 512, 0), ("i8", "dots", 65, 1_048_576, 512, 32), ("i8", "dots", 128, 131_040, 512, 0), ("i8", "dots", 128, 131_072, 512, 32),
    ("i8", "dots", 255, 122_880, 512, 0), ("i8", "dots", 255, 122_912, 512, 32), ("i8", "angular", 160, 500_000, 768, 0), ("i8", "angular", 161, 500_000, 768, 32),
    ("f16", "dots", 128, 500_000, 500, 32), ("f16", "dots", 129, 500_001, 500, 32), ("f16", "dots", 128, 500_001, 500, 0), ("f16", "dots", 128, 500_001, 600, 32), ("i8", "dots", 128, 500_001, 1000, 32),
    ("i8", "dots", 1000, 300_001, 700, 32),
    ("i8", "dots", 512, 262_112, 256, 32), ("i8", "dots", 512, 262_144, 256, 64), ("i8", "dots", 256, 500_000, 256, 32), ("i8", "dots", 257, 500_000, 256, 64),
    ("bf16", "dots", 512, 500_000, 256, 32), ("bf16", "dots", 513, 500_000, 256, 64), ("u8", "dots", 768, 500_000, 768, 32), ("u8", "dots", 769, 500_000, 768, 64),
    ("u8", "dots", 1024, 109_216, 768, 32), ("u8", "dots", 1024, 109_248, 768, 64), ("u8", "dots", 1024, 500_001, 768, 32), ("f16", "dots", 1024, 500_000, 350, 32)])
def test_where_a_is_kept(dtype, metric, m, n, k, rows):
    assert resident_of(dtype, metric, m, n, k)[0] == rows


# Rows of C a multiple of 4 KiB apart: strips of 33 tiles in the place of 32, up to 129; tiles where too many rows share them.
@pytest.mark.parametrize("dtype, metric, m, n, k, tiles", [
    ("i8", "dots", 2048, 32_768, 512, 33), ("i8", "dots", 2048, 32_736, 512, 32), ("i8", "euclidean", 4982, 12_288, 256, 33), ("i8", "dots", 4982, 12_288, 768, 33),
    ("i8", "dots", 4982, 12_288, 256, 0), ("i8", "dots", 4982, 12_288, 512, 0), ("e2m3", "dots", 4982, 12_288, 512, 33), ("u8", "dots", 4982, 12_288, 512, 33), ("u8", "dots", 4982, 12_288, 256, 0), ("i8", "dots", 4982, 12_256, 256, 32), ("i8", "euclidean", 8192, 16_384, 256, 64), ("bf16", "dots", 60_000, 1024, 256, 0), ("bf16", "dots", 60_000, 1024, 600, 32),
    ("i8", "angular", 2048, 131_072, 768, 129), ("i8", "angular", 2048, 163_840, 768, 160), ("i8", "dots", 1024, 1_048_576, 768, 256)])
def test_strips_out_of_step(dtype, metric, m, n, k, tiles):
    assert resident_of(dtype, metric, m, n, k)[2] == tiles
