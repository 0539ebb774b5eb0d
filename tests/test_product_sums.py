"""Order of a fused product's fp32 additions: a lane sums each 16-byte vector
of weights from zero and adds that to its running sum, so a lane's chain is a
vector's products plus one addition per vector, not all of its products; and the activations' place."""
import subprocess
from pathlib import Path

import numpy as np
import pytest
import torch

from neuralzip_amd import _native
from neuralzip_amd.dtypes import DTYPES
from nz_helpers import Encoded, singleton_header
from test_matvec import run_matvec
from test_row_products import run_rows

CSRC = Path(__file__).resolve().parents[1] / "neuralzip_amd" / "csrc"


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


def test_activation_offsets_hold_for_rows_of_nearly_four_gigabytes(tmp_path):
    """nz_activation_offset for every vector of a tile that crosses the end of
    its row, against 64-bit arithmetic: short rows, and rows so long that the
    offset of the next row's first columns passes 2^32 before a row is taken off."""
    probe, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    probe.write_text("""
#include <cstdio>
#include <initializer_list>
#include "nz_format.h"
int main() {
    const uint32_t widths[] = {2, 4};
    for (uint32_t es : widths)
        for (uint64_t row : {4096ull, 28672ull, 0x7FFFFFF0ull, 0xFFFFF000ull, 0xFFFFFFF0ull})   // bytes
            for (uint32_t left = 16; left <= 4096; left += 16) {                                // bytes left in the first row
                const uint32_t col0 = static_cast<uint32_t>((row - left) / es);
                for (uint32_t i = 0; i < 2048; i += 16 / es) {
                    const uint64_t byte = row - left + uint64_t(i) * es, want = byte >= row ? byte - row : byte;
                    if (want >= row) continue;
                    const uint32_t got = nz_activation_offset(col0 * es + i * es - static_cast<uint32_t>(row), static_cast<uint32_t>(row));
                    if (got != want) return std::printf("row %llu left %u element %u: %u\\n",
                                                        (unsigned long long)row, left, i, got), 1;
                }
            }
    return 0;
}
""")
    try:
        subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), str(probe), "-o", str(exe)], check=True,
                       capture_output=True, text=True)
    except FileNotFoundError:
        pytest.skip("no C++ compiler for the probe")
    result = subprocess.run([str(exe)], capture_output=True, text=True)
    assert result.returncode == 0, result.stdout
