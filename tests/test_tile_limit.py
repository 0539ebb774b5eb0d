"""Tiles stage at most 2048 elements of 16-bit words and 1024 of 32-bit ones
(four merge rounds), the elements of its first vector ahead of a tile's first
one included: sizes around the rounds and around a second tile, at aligned and
odd places of the workspace, with codes short enough for the limit to bind and
long enough for 64 windows to bind."""
import numpy as np
import pytest
import torch

from neuralzip_amd import _native
from neuralzip_amd.dtypes import DTYPES
from nz_helpers import Encoded, singleton_header
from test_layout_emulator import emulate_case

LIMIT = {torch.bfloat16: 2048, torch.float16: 2048, torch.float32: 1024}
OFFSETS = (8, 3, 7)


def words_of(kind, n, dtype):
    g = torch.Generator().manual_seed(n)
    if kind == "limit":     # one bit per exponent or so
        return torch.where(torch.rand(n, generator=g) < 0.9, 0.5, 0.01).to(dtype)
    return torch.randn(n, generator=g).mul(0.02).to(dtype)


SIZES = (1, 511, 513, 1023, 1025, 1535, 1536, 1537, 1600, 2047, 2048, 2049, 3071, 3073, 4095, 4097, 10001)


def case_of(kind, n, dtype, offset):
    raw = words_of(kind, n, dtype).view(torch.uint8).numpy().copy()
    book = _native.Codebook(singleton_header(words_of(kind, 40000, dtype).view(torch.uint8).numpy(), dtype, prior=1))
    return [(raw, dtype, 1 << 20, [0], offset)], {0: book}


@pytest.mark.parametrize("offset", OFFSETS)
@pytest.mark.parametrize("dtype", sorted(LIMIT, key=str))
@pytest.mark.parametrize("kind", ["limit", "windows"])
def test_tiles_hold_at_most_four_rounds(kind, dtype, offset):
    vector, limit = 16 // DTYPES[dtype].element_size, LIMIT[dtype]
    for n in SIZES:
        tensors, books = case_of(kind, n, dtype, offset)
        _, _, tiles = Encoded(tensors, books).host_image()
        ahead = (offset + tiles["out0"].astype(int)) % vector
        assert (ahead + tiles["n_out"]).max() <= limit and tiles["n_out"].astype(int).sum() == n
        if kind == "limit" and n > limit + 64:     # the limit binds, but for the line its end is cut back to
            assert tiles["n_out"].max() > limit - 64
        emulate_case(tensors, books, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", sorted(LIMIT, key=str))
@pytest.mark.parametrize("kind", ["limit", "windows"])
@pytest.mark.parametrize("n", SIZES)
def test_tiles_of_four_rounds_decode(kind, n, dtype):
    from test_gpu_decode import check_case
    for offset in OFFSETS:
        tensors, books = case_of(kind, n, dtype, offset)
        check_case(tensors, books, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 2, 3, 4])
@pytest.mark.parametrize("dtype", sorted(LIMIT, key=str))
@pytest.mark.parametrize("elements", [8, 512, 1016, 1024, 1032, 1528, 1536, 1544, 2040, 2048])
def test_products_of_tiles_that_end_around_each_round(elements, dtype, batch):
    """One tile per chunk of `elements` (two where 32-bit words exceed their
    limit), across the ends of rows, both ways of adding the tiles up."""
    from test_matvec import check_product, run_matvec
    from test_row_products import run_rows
    rows, cols = 9, 2048
    w = words_of("limit", rows * cols, dtype).view(rows, cols)
    raw = w.view(torch.uint8).numpy().reshape(-1).copy()
    books = {0: _native.Codebook(singleton_header(raw, dtype, prior=1))}
    base, descs, tiles = Encoded([(raw, dtype, elements, [0] * -(-w.numel() // elements), 64)], books).host_image()
    assert elements > LIMIT[dtype] or tiles["n_out"][0] == elements
    x = torch.randn(batch, cols, generator=torch.Generator().manual_seed(batch)).to(dtype)
    (two,) = run_matvec(base, descs, tiles, dtype, [(64, rows)], cols, x, calls=1)
    check_product(two[0], w, x, None, dtype)
    (one,) = run_rows(base, descs, tiles, dtype, [(64, rows)], cols, x, [None], 64, 1.0)
    assert torch.equal(one.view(torch.uint8), two[0].view(torch.uint8))
