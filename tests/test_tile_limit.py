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


@pytest.mark.parametrize("dtype", sorted(LIMIT, key=str))
@pytest.mark.parametrize("offset", [64, 67])
def test_planners_refuse_coded_tiles_past_the_staging_area(dtype, offset):
    """Tiles of a caller's own that a wavefront's staging area does not hold:
    the record and row planners know the word's size and the tile's place in
    its first vector, the launch planners only that no tile holds over 2048.
    Raw tiles are not staged."""
    es = DTYPES[dtype].element_size
    limit, ahead = LIMIT[dtype], offset % (16 // es)
    cols = 4096
    descs, tiles = np.zeros(1, _native.FRAG_DESC), np.zeros(3, _native.TILE)
    descs["kind"], descs["out"], descs["lane_stride"] = _native.KIND_SHORT, offset, 8192
    weights = [(offset - ahead, 2)]

    def plans(sizes):
        tiles["n_out"], tiles["out0"] = sizes, np.concatenate([[0], np.cumsum(sizes)[:-1]])
        _native.matvec_plan(descs, tiles, weights, cols, es)

    def records(sizes):
        tiles["n_out"], tiles["out0"] = sizes, np.concatenate([[0], np.cumsum(sizes)[:-1]])
        _native.matvec_tiles(descs, tiles, weights, cols, es, 1 << 20)

    for call in (plans, records):
        with pytest.raises(_native.NativeError, match="staging area"):
            call((limit - ahead + 1, 100, 100))
        with pytest.raises(_native.NativeError, match="exactly once"):     # accepted so far
            call((limit - ahead, 100, 100))
    for call in (lambda: _native.plan_work(descs, tiles, 4), lambda: _native.plan_work_interleaved(descs, tiles, 4)):
        descs["kind"] = _native.KIND_SHORT
        tiles["n_out"] = (2049, 100, 100)
        with pytest.raises(_native.NativeError, match="staging area"):
            call()
        descs["kind"] = _native.KIND_RAW
        call()
        descs["kind"], tiles["n_out"] = _native.KIND_SHORT, (2048, 100, 100)
        call()


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
