"""128 x 128 tiles of i8 whose A goes straight into LDS: the same bits as staged through registers."""
import numpy as np
import pytest
import torch

import numkong_amd as nk
from tests.test_strips_gpu import framed, through, untouched
from tests.test_unaligned_gpu import DEV, values_of

pytestmark = pytest.mark.gpu


# The fewest rows and stages that go this way, depths short of whole stages (rows on 16 bytes all the same), tiles cut off by both
# edges, more tiles than workgroups are resident.
@pytest.mark.parametrize("m, n, k, after", [(257, 1, 3072, 0), (384, 128, 3584, 0), (300, 1000, 3057, 1), (2048, 2048, 4096, 0), (513, 129, 8192, 3), (4097, 4100, 3500, 0)])
def test_same_bits_as_staged(m, n, k, after):
    rng = np.random.default_rng(95)
    wide = values_of("i8", m, (k + 15) // 16 * 16, rng).to(DEV)
    a, packed = wide[:, :k], nk.dots_pack(values_of("i8", n, k, rng).to(DEV), "i8")
    expected = through(3 | 1 << 30, lambda: nk.dots_packed(a, packed))
    whole, window = framed(m, n, 0, after, torch.int32)
    through(3, lambda: nk.dots_packed(a, packed, out=window))
    assert torch.equal(window.contiguous(), expected)
    assert torch.equal(expected[::97, ::31].cpu().long(), a[::97].cpu().long() @ values_of("i8", n, k, _again(m, k))[::31].long().T)
    assert untouched(whole, m, n, 0)


def _again(m, k):
    """The generator as it stood when B was drawn."""
    rng = np.random.default_rng(95)
    values_of("i8", m, (k + 15) // 16 * 16, rng)
    return rng


# Windows of all pairs whose first row is not one of the image's tiles take A from the vectors: the same tile, along a triangle's list.
@pytest.mark.parametrize("start, count, k", [(33, 1000, 3072), (1, 700, 3584), (95, 1300, 4096)])
def test_windows_of_all_pairs(start, count, k):
    rng = np.random.default_rng(99)
    vectors = values_of("i8", count, k, rng).to(DEV)

    def window(config):
        out = torch.full((count, count), 77, dtype=torch.int32, device=DEV)
        return through(config, lambda: nk.dots_symmetric(vectors, "i8", out=out, start_row=start, end_row=count))

    straight = window(3)
    assert torch.equal(straight, window(3 | 1 << 30))
    expected = (vectors.cpu().double() @ vectors.cpu().double().T).to(torch.int32)  # (exact: whole numbers below 2^53)
    row, column = torch.arange(count)[:, None], torch.arange(count)[None, :]
    assert torch.equal(straight.cpu(), torch.where((row >= start) & (column >= row), expected, 77))
