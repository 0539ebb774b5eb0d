"""Decode workgroups with fewer, as many and more tiles than wavefronts
(a wavefront's first tile is the one of its index, the others are claimed),
at odd fragment ends, whose partial vectors' raw bytes are loaded apart."""
import numpy as np
import pytest
import torch

from neuralzip_amd import _native
from nz_helpers import Encoded, singleton_header
from test_gpu_decode import check_case


@pytest.mark.gpu
@pytest.mark.parametrize("flags", [0, _native.DECODE_HALF_GROUPS, _native.DECODE_CACHED_STORES])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("tiles", [1, 7, 8, 9, 16, 17, 40])
def test_workgroups_of_few_tiles(tiles, dtype, flags):
    g = torch.Generator().manual_seed(tiles)
    words = (torch.randn(tiles * 2048, generator=g) * 0.02).to(dtype)
    book = _native.Codebook(singleton_header(words.view(torch.uint8).numpy(), dtype))

    def tensors(n):
        return [(words[:n].view(torch.uint8).numpy().copy(), dtype, n, [0], 3)]

    def count(n):
        return len(Encoded(tensors(n), {0: book}).host_image()[2])

    low, high = 1, words.numel()     # the largest odd size of that many tiles
    while high - low > 1:
        mid = (low + high) // 2
        low, high = (mid, high) if count(mid) <= tiles else (low, mid)
    n = low - 1 + low % 2
    assert count(n) == tiles
    check_case(tensors(n), {0: book}, dtype, slots=1, interleaved=True, flags=flags)


@pytest.mark.gpu
@pytest.mark.parametrize("flags", [0, _native.DECODE_HALF_GROUPS, _native.DECODE_CACHED_STORES])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_empty_segments_decode_nothing(dtype, flags, monkeypatch):
    """Segments without tiles, which a caller's own plan may hold: before,
    between and behind the others, the last past the end of the tile list."""
    plan_work = _native.plan_work

    def with_empty_segments(descs, tiles, slots):
        segments = plan_work(descs, tiles, slots)
        empty = segments[:1].copy()
        parts = []
        for at in (0, segments["tile1"][0], len(tiles)):
            empty["tile0"] = empty["tile1"] = at
            parts.append(empty.copy())
        return np.concatenate([parts[0], segments[:1], parts[1], segments[1:], parts[2]])

    monkeypatch.setattr(_native, "plan_work", with_empty_segments)
    words = (torch.randn(50001, generator=torch.Generator().manual_seed(2)) * 0.02).to(dtype)
    raw = words.view(torch.uint8).numpy().copy()
    check_case([(raw, dtype, 20000, [0, -1, 0], 3)], {0: _native.Codebook(singleton_header(raw, dtype))}, dtype, slots=4,
               flags=flags)
