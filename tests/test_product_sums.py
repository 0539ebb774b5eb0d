"""Order of a fused product's fp32 additions: a lane sums each 16-byte vector
of weights from zero and adds that to its running sum, so a lane's chain is a
vector's products plus one addition per vector, not all of its products."""
import numpy as np
import pytest
import torch

from neuralzip_amd import _native
from neuralzip_amd.dtypes import DTYPES
from nz_helpers import Encoded, singleton_header
from test_matvec import run_matvec
from test_row_products import run_rows


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_a_vectors_products_are_summed_before_they_join_the_lanes_sum(dtype, batch):
    """Lane 0 holds 2^25 (one product of its first vector) when its second
    vector's products, ones, arrive: each of them (and a pair of them) is half
    a unit in the last place or less and would be lost, their sum of 4 or 8 is
    not. Lane 1 holds -2^25, so that the row's sum is exactly that sum."""
    V, cols, rows = 16 // DTYPES[dtype].element_size, 2048, 4
    w = torch.zeros(rows, cols)
    w[:, 0], w[:, V] = 2.0 ** 12, -2.0 ** 12
    w[:, 64 * V:65 * V] = 1.0
    x = torch.ones(batch, cols)
    x[:, [0, V]] = 2.0 ** 13
    w, x = w.to(dtype), x.to(dtype)
    raw = w.view(torch.uint8).numpy().reshape(-1).copy()
    books = {0: _native.Codebook(singleton_header(raw, dtype))}
    base, descs, tiles = Encoded([(raw, dtype, cols, [0] * rows, 64)], books).host_image()   # a row's first tile starts with it
    weights = [(64, rows)]
    (two,) = run_matvec(base, descs, tiles, dtype, weights, cols, x, calls=1)
    (one,) = run_rows(base, descs, tiles, dtype, weights, cols, x, [None], 64, 1.0)
    for y in (two[0], one):
        assert np.array_equal(y.float().numpy(), np.full((batch, rows), V, np.float32))
