"""f32 and f64 products of few rows, and of few tiles, run through tiles of fewer rows: the same bits as through the largest."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from numkong_amd import api
from tests import support

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CALLS = (nk.dots_packed, nk.angulars_packed, nk.euclideans_packed)


def same(x, y):
    return torch.equal(x.view(torch.int64), y.view(torch.int64))


# Row counts around every tile's edge (4, 16, 32, 64, 128); depths under, at and around the 8 and 32 of a step. A result
# does not depend on how many other rows are asked for, so the rows of a tall call, which takes 64 rows to a tile (20,000
# columns give it more than enough tiles; f32 takes 128 only beyond 512 values, below), are what the short calls must
# return, bit for bit.
@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("depth", [1, 7, 32, 97, 300])
def test_few_rows_give_the_bits_of_the_largest_tile(dtype, depth):
    rng = np.random.default_rng(51)
    a = torch.from_numpy(rng.standard_normal((512, depth)).astype(support.STORAGE[dtype])).to(DEV)
    b = torch.from_numpy(rng.standard_normal((20000, depth)).astype(support.STORAGE[dtype])).to(DEV)
    packed = nk.dots_pack(b, dtype)
    few = nk.dots_pack(b[:70], dtype)
    for call in CALLS:
        tall = call(a, packed)
        for rows in (1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 63, 64, 65, 128, 129, 193):
            assert same(call(a[:rows], packed), tall[:rows]), f"{call.__name__} {rows} rows"
            assert same(call(a[:rows], few), tall[:rows, :70].contiguous()), f"{call.__name__} {rows} rows, 70 columns"


# A shape for every tile: the row count at which the rule picks it on 256 compute units, by the costs of f32_tile_rows (deeper
# than 512 values) and f64_tile_rows over the 64 column tiles of 4090 vectors. f32: 505 rows are 256 tiles of 128 (8.2 against
# two rounds of 64 at 4.2 each), 250 rows 256 tiles of 64 (4.2 against two rounds of 32 at 2.75), 120 rows 256 of 32 (2.75
# against two rounds of 16 at 2.6), 60 rows 256 of 16 (2.6 against 2.75). f64: 250 rows 256 tiles of 64 (4.0 against four
# rounds of 16 at 1.03), 60 rows 256 of 16 (1.03 against four rounds of 4 at 0.32), 12 rows 192 of 4. Ragged rows, columns and
# depths (one whole step or a part of it at the end), A in wider rows that start off every 16-byte boundary and aligned; an
# image of another depth poisons every output and touches nothing else.
# Up to 512 values the 505 rows take 128 (more than 256 values, or a distance) where 1100 rows, two rounds of it, take 64.
DEEP = (517, 544)
TILES = [("f32", 128, 505, DEEP), ("f32", 64, 250, DEEP), ("f32", 32, 120, DEEP), ("f32", 16, 60, DEEP), ("f32", 128, 505, (257, 512)), ("f32", 64, 1100, (257, 512)),
         ("f64", 64, 250, DEEP), ("f64", 16, 60, DEEP), ("f64", 4, 12, DEEP)]


@pytest.mark.parametrize("dtype, tile, m, depths", TILES)
def test_every_tile_against_the_oracle(oracle, dtype, tile, m, depths):
    rng = np.random.default_rng(53)
    n = 4090
    sampled = np.unique(np.r_[0:3, tile // 2 - 1:tile // 2 + 2, tile - 1:min(tile + 2, m), m - 3:m].clip(0, m - 1))
    for k in depths:
        a, b = support.random_matrix(oracle, dtype, m, k, rng, "lognormal"), support.random_matrix(oracle, dtype, n, k, rng, "lognormal")
        a[1], b[2], b[n - 1] = 0, a[m - 1], a[0]  # a zero row; identical rows, one of them in the ragged last tile
        gb = torch.from_numpy(b).to(DEV)
        packed, other = nk.dots_pack(gb, dtype), nk.dots_pack(gb[:, 1:].contiguous(), dtype)
        norms = oracle.row_sumsq(dtype, a[sampled])[:, None] + oracle.row_sumsq(dtype, b)[None, :]
        for pad, offset in ((0, 0), (3, 1)):
            rows = torch.full((m, k + pad + offset), float("nan"), dtype=gb.dtype, device=DEV)[:, offset:offset + k]
            rows.copy_(torch.from_numpy(a))
            where = f"{dtype} {tile} rows, {m}x{n}x{k} pad {pad} offset {offset}"
            got = nk.dots_packed(rows, packed).cpu().numpy()[sampled]
            assert np.array_equal(got.view(np.uint64), oracle.dots_packed(dtype, a[sampled], b).view(np.uint64)), where
            for metric, call in (("angular", nk.angulars_packed), ("euclidean", nk.euclideans_packed)):
                got = call(rows, packed).cpu().numpy()[sampled]
                assert np.isfinite(got).all(), f"{metric} {where}"
                assert support.wide_distances_agree(metric, got, oracle.spatials_packed(metric, dtype, a[sampled], b), norms), f"{metric} {where}"
            for kind in (support.KIND_PACKED, support.KIND_ANGULARS, support.KIND_EUCLIDEANS):
                out = torch.full((m, n + 1), -7.0, dtype=torch.float64, device=DEV)
                arguments = (api.DTYPES[dtype][0], rows.data_ptr(), other.buffer.data_ptr(), out.data_ptr(), m, n, k,
                             rows.stride(0) * rows.element_size(), (n + 1) * 8, torch.cuda.current_stream().cuda_stream)
                lib = nk.library()
                status = lib.nk_amd_dots_packed_async(*arguments) if kind == support.KIND_PACKED else lib.nk_amd_spatials_packed_async(kind, *arguments)
                torch.cuda.synchronize()
                assert status == 0 and (out[:, n] == -7.0).all() and (out[:, :n].contiguous().view(torch.int64) == -1).all(), where


# All pairs of 4000 vectors: as many tiles as whole rounds of the largest tile hold (f32: 1024 of 128 rows, 4 rounds at 8.2
# against 16 of 32 rows at 2.3; f64: 2016 of 64 rows, 8 rounds at 4.0 against 32 of 16 rows at 1.03), on rows around the
# tiles' edges.
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_largest_tile_of_all_pairs(oracle, dtype):
    rng = np.random.default_rng(54)
    count, depth = 4000, 70
    vectors = support.random_matrix(oracle, dtype, count, depth, rng, "lognormal")
    squares = oracle.row_sumsq(dtype, vectors)
    on_gpu = torch.from_numpy(vectors).to(DEV)
    for metric, call in (("dots", nk.dots_symmetric), ("angular", nk.angulars_symmetric), ("euclidean", nk.euclideans_symmetric)):
        out = torch.full((count, count), -7.0, dtype=torch.float64, device=DEV)
        call(on_gpu, dtype, out=out)
        for start, rows in ((0, 2), (63, 2), (127, 2), (2047, 2), (3998, 2)):
            got = out[start:start + rows].cpu().numpy()
            serial = oracle.symmetric(metric, dtype, vectors, start, rows)[start:start + rows]
            own = np.arange(count)[None, :] >= np.arange(start, start + rows)[:, None]
            assert (got[~own] == -7.0).all()
            if metric == "dots":
                assert np.array_equal(got[own].view(np.uint64), serial[own].view(np.uint64)), (dtype, start)
            else:
                norms = (squares[start:start + rows, None] + squares[None, :])[own]
                assert support.wide_distances_agree(metric, got[own], serial[own], norms), (dtype, metric, start)


# All pairs of few vectors: fewer tiles of the largest size than compute units, windows of rows among them.
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_few_tiles_of_all_pairs(dtype):
    oracle = support.load_oracle()
    rng = np.random.default_rng(52)
    for count, depth, start, rows in ((5, 9, 0, 5), (65, 40, 0, 65), (257, 33, 0, 257), (300, 64, 99, 3), (700, 31, 333, 70)):
        vectors = rng.standard_normal((count, depth)).astype(support.STORAGE[dtype])
        out = torch.full((count, count), -7.0, dtype=torch.float64, device=DEV)
        nk.dots_symmetric(torch.from_numpy(vectors).to(DEV), dtype, out=out, start_row=start, end_row=start + rows)
        expected = np.full((count, count), -7.0)
        serial = oracle.symmetric("dots", dtype, vectors, start, rows)
        row, column = np.indices((count, count))
        own = (row >= start) & (row < start + rows) & (column >= row)
        expected[own] = serial[own]
        assert np.array_equal(out.cpu().numpy().view(np.uint64), expected.view(np.uint64)), (count, depth, start)


# Rows of a multiple of four values at 16-byte addresses (read whole, to the last step of 32 values) against the same values at
# other addresses (read one by one); depths around the groups of 16 and the steps of 32, which the last step's second group may
# lie behind. NaN behind every row.
@pytest.mark.parametrize("metric", ["dots", "angular", "euclidean"])
def test_f32_rows_of_whole_quads(metric):
    call = {"dots": nk.dots_packed, "angular": nk.angulars_packed, "euclidean": nk.euclideans_packed}[metric]
    rng = np.random.default_rng(57)
    for depth in (4, 12, 16, 20, 32, 36, 48, 52, 64, 80, 100, 112, 300):
        packed = nk.dots_pack(torch.from_numpy(rng.standard_normal((97, depth)).astype(np.float32)).to("cuda:0"), "f32")
        for rows in (3, 40, 130):
            values = torch.from_numpy(rng.standard_normal((rows, depth)).astype(np.float32)).to("cuda:0")
            results = []
            for pad, offset in ((4, 0), (4, 1)):
                whole = torch.full((rows, depth + pad), float("nan"), device="cuda:0")
                view = whole[:, offset:offset + depth]
                view.copy_(values)
                results.append(call(view, packed))
            assert torch.equal(results[0].view(torch.int64), results[1].view(torch.int64)), f"{metric} {rows} rows of {depth}"


# The quicker root of the f32 distances gives way where a sum of squares is zero, infinite, NaN or near the ends of f64's range: the
# f64 kernel, which always takes the reference's form, has the expected values (the products of these vectors are exact).
@pytest.mark.parametrize("metric", ["angular", "euclidean"])
def test_f32_distances_of_extreme_vectors(metric):
    call = {"angular": nk.angulars_packed, "euclidean": nk.euclideans_packed}[metric]
    inf, nan = float("inf"), float("nan")
    rows = [[0, 0, 0, 0], [1e-45, 0, 0, 0], [1e-42, -1e-42, 0, 0], [3e38, 0, 0, 0], [3e38, -3e38, 3e38, 3e38], [inf, 0, 0, 0], [-inf, 1, 0, 0],
            [nan, 1, 2, 3], [1, 2, 3, 4], [-4, 3, 0.5, -1], [1e-20, 0, 1e-20, 0], [0, 1e19, 0, 0]]
    values = torch.tensor(rows * 6, dtype=torch.float32, device="cuda:0")
    got = call(values, nk.dots_pack(values, "f32"))
    expected = call(values.double(), nk.dots_pack(values.double(), "f64"))
    assert torch.equal(got.isnan(), expected.isnan()) and torch.equal(got.isinf(), expected.isinf())
    finite = expected.isfinite()
    # (roundings of a few units of 2^-53: of one for the angular distance, of the result for the other)
    scale = torch.ones_like(expected) if metric == "angular" else expected.abs()
    assert bool(((got - expected).abs()[finite] <= 16 * 2.0**-53 * scale[finite]).all())


# Both orders of walking over the tiles of a product, on both sides of where the depth and the rows of tiles switch between them (64 and
# 96 values; three and eight rows of tiles of 64), a last band of one row of tiles and of all sixteen: the rows of a product are those of
# the products of 64 of them, which are one row of tiles.
@pytest.mark.parametrize("depth", [64, 65, 96, 97])
def test_f32_walks(depth):
    rng = np.random.default_rng(98)
    a = torch.from_numpy(rng.standard_normal((2112, depth)).astype(np.float32)).to(DEV)
    packed = nk.dots_pack(torch.from_numpy(rng.standard_normal((5003, depth)).astype(np.float32)).to(DEV), "f32")
    for call in CALLS:
        single = torch.cat([call(a[first:first + 64], packed) for first in range(0, 2112, 64)])
        for rows in (65, 192, 193, 512, 513, 1024, 1025, 2048, 2112):
            out = torch.full((rows + 1, 5003), -7.0, dtype=torch.float64, device=DEV)
            call(a[:rows], packed, out=out[:rows])
            assert same(out[:rows], single[:rows]), f"{call.__name__} {rows} rows"
            assert bool((out[rows] == -7.0).all())
