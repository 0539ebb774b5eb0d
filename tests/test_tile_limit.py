"""Tiles of 16-bit words stage at most 1536 elements (three merge rounds):
sizes around one, two and three rounds and around a second tile, with codes
short enough for the limit to bind and long enough for 64 windows to bind."""
import numpy as np
import pytest
import torch

from neuralzip_amd import _native
from nz_helpers import Encoded, singleton_header
from test_layout_emulator import emulate_case


def words_of(kind, n):
    g = torch.Generator().manual_seed(n)
    if kind == "limit":     # one bit per exponent or so
        return torch.where(torch.rand(n, generator=g) < 0.9, 0.5, 0.01).bfloat16()
    return torch.randn(n, generator=g).mul(0.02).bfloat16()


SIZES = (1, 511, 513, 1023, 1025, 1535, 1536, 1537, 1600, 3071, 3073, 10001)


def case_of(kind, n):
    raw = words_of(kind, n).view(torch.uint8).numpy().copy()
    book = _native.Codebook(singleton_header(words_of(kind, 40000).view(torch.uint8).numpy(), torch.bfloat16, prior=1))
    return [(raw, torch.bfloat16, 1 << 20, [0], 8)], {0: book}


@pytest.mark.parametrize("kind", ["limit", "windows"])
@pytest.mark.parametrize("n", SIZES)
def test_tiles_hold_at_most_three_rounds(kind, n):
    tensors, books = case_of(kind, n)
    _, _, tiles = Encoded(tensors, books).host_image()
    assert tiles["n_out"].max() <= 1536 and tiles["n_out"].astype(int).sum() == n
    if kind == "limit" and n > 1536:
        assert tiles["n_out"].max() > 1536 - 64
    emulate_case(tensors, books, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["limit", "windows"])
@pytest.mark.parametrize("n", SIZES)
def test_tiles_of_three_rounds_decode(kind, n):
    from test_gpu_decode import check_case
    tensors, books = case_of(kind, n)
    check_case(tensors, books, torch.bfloat16)
