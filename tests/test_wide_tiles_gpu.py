"""f32 and f64 products of few rows, and of few tiles, run through tiles of fewer rows: the same bits as through the largest."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests import support

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
CALLS = (nk.dots_packed, nk.angulars_packed, nk.euclideans_packed)


def same(x, y):
    return torch.equal(x.view(torch.int64), y.view(torch.int64))


# Row counts around every tile's edge (4, 16, 32, 64, 128); depths under, at and around the 8 and 32 of a step. A result
# does not depend on how many other rows are asked for, so the rows of a tall call, which takes the largest tile (20,000
# columns give it more than enough tiles), are what the short calls must return, bit for bit.
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
