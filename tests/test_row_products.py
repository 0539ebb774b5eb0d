"""Fused products in one launch: row segments (nz_matvec_row_plan), whose
workgroups own whole output rows and add up their partial sums themselves
(nz_matvec_rows). The bar is the two-launch form: the same bits."""
import numpy as np
import pytest
import torch

from neuralzip_amd import _native
from neuralzip_amd.dtypes import DTYPES
from nz_helpers import Encoded, segment_lengths, singleton_header
from test_matvec import encoded_case, launch_order, long_code_weight, random_weight, run_matvec

CASES = ("one-row", "odd-rows", "two-books", "raw-rows", "wide", "many", "long")


def case_of(name, dtype):
    """(base, descs, tiles, [(offset, rows)], cols): weights whose chunks end
    at rows, so that a row plan exists."""
    offset, vector = 64, 16 // DTYPES[dtype].element_size
    shapes = {"one-row": [(1, 2048)], "odd-rows": [(37, 2048 + 3 * vector), (5, 2048 + 3 * vector)],
              "two-books": [(40, 4096), (24, 4096)], "raw-rows": [(16, 4096), (16, 4096)], "wide": [(11, 16384)],
              "many": [(700, 2048), (1, 2048), (331, 2048)], "long": [(12, 4096)]}[name]
    tensors, books, weights, cols = [], {}, [], shapes[0][1]
    for i, (rows, _) in enumerate(shapes):
        w = long_code_weight(rows, cols, 3) if name == "long" else random_weight(dtype, rows, cols, seed=20 + i)
        raw = w.view(torch.uint8).numpy().reshape(-1).copy()
        if name == "long":
            books[i] = _native.Codebook(b"NZM1" + segment_lengths(56), bytes((127, 127, 125, 126)))
        elif i == 0 or name == "two-books":
            books[i] = _native.Codebook(singleton_header(raw, dtype))
        book = -1 if name == "raw-rows" and i else i if i in books else 0
        step = 8 * cols if rows % 8 == 0 else rows * cols
        tensors.append((raw, dtype, step, [book] * -(-w.numel() // step), offset))
        weights.append((offset, rows))
        offset += -(-w.numel() // 256) * 256 + 256
    base, descs, tiles = Encoded(tensors, books).host_image()
    return base, descs, launch_order(descs, tiles), weights, cols


@pytest.mark.parametrize("slots,weight", [(1, 1.0), (6, 1.75), (64, 1.0), (512, 1.75)])
@pytest.mark.parametrize("name", CASES)
def test_row_segments_hold_every_sum_of_their_rows_once(name, slots, weight):
    dtype = torch.bfloat16
    base, descs, tiles, weights, cols = case_of(name, dtype)
    row_index, entries = _native.matvec_plan(descs, tiles, weights, cols, 2)
    segments, words = _native.matvec_row_plan(descs, tiles, row_index, entries, cols, slots, weight)
    records = _native.matvec_tiles(descs, tiles, weights, cols, 2, base.size)
    assert len(segments) and segments["row0"][np.argsort(segments["row0"])][0] == 0
    owned = np.zeros(len(row_index) - 1, int)
    for s in segments:
        owned[s["row0"]:s["row1"]] += 1
        assert s["entry0"] == row_index[s["row0"]] and s["entry0"] + s["entries"] == row_index[s["row1"]]
        written = np.zeros(s["entries"], int)
        for t in range(s["tile0"], s["tile1"]):
            f, lut = descs[tiles[t]["frag"]], descs[s["lut_frag"]]["lut"]
            assert f["kind"] == s["kind"] and (f["kind"] == _native.KIND_RAW or f["lut"] == lut)
            end = int(records[t]["head"] & 15) + int(tiles[t]["n_out"])
            for slot in range(1 + (cols - int(records[t]["col0"]) < end)):
                at = int(records[t]["entry"]) + slot - int(s["entry0"])
                if 0 <= at < len(written):
                    written[at] += 1
        assert (written == 1).all()
    assert (owned == 1).all()
    rows = (segments["row1"] - segments["row0"]).astype(int)
    assert words == tuple(int((rows + 1 + segments["entries"].astype(int) * n).max()) for n in (1, 2, 4))


def test_no_row_plan_where_codebooks_change_inside_rows():
    w, enc, offset = encoded_case("nzm1", torch.bfloat16)     # chunks of 9.14 rows, two codebooks in turn
    _, descs, tiles = enc.host_image()
    tiles = launch_order(descs, tiles)
    plan = _native.matvec_plan(descs, tiles, [(offset, w.shape[0])], w.shape[1], 2)
    segments, _ = _native.matvec_row_plan(descs, tiles, *plan, w.shape[1], 512)
    assert not len(segments)


def plain_tiles(rows, cols, elements, chunk=None, books=1, kind=_native.KIND_SHORT):
    """Descriptors and launch-ordered tiles of a rows x cols weight in chunks
    whose codebooks take turns: what the planners read of them."""
    total, chunk = rows * cols, chunk or rows * cols
    starts = np.arange(0, total, chunk)
    descs = np.zeros(len(starts), _native.FRAG_DESC)
    descs["kind"], descs["out"], descs["lut"] = kind, starts, np.arange(len(starts)) % books * 65536
    tiles = []
    for f, start in enumerate(starts):
        size = min(chunk, total - start)
        t = np.zeros(-(-size // elements), _native.TILE)
        t["frag"], t["out0"] = f, np.arange(0, size, elements)
        t["n_out"] = np.minimum(elements, size - t["out0"].astype(int))
        tiles.append(t)
    return descs, launch_order(descs, np.concatenate(tiles))


@pytest.mark.parametrize("rows,cols,elements,chunk,books,slots,whole", [
    # few rows of very many columns: whole rows would be a few workgroups of a million elements
    (1, 1 << 20, 1600, None, 1, 512, False), (4, 131072, 1600, None, 1, 512, False),
    (64, 65536, 1024, None, 1, 512, False), (64, 53248, 1600, None, 1, 512, False),
    # codebooks that change after every few rows: more row segments than the device runs at once,
    # as many as it runs, and (uneven) a few fewer
    (34 * 32, 4096, 1600, 131072, 2, 32, False), (32 * 32, 4096, 1600, 131072, 2, 32, True),
    (20 * 32, 4096, 1600, 131072, 2, 32, False), (34 * 2, 4096, 1600, 8192, 2, 32, False),
    # short and long rows that divide evenly enough
    (6144, 4096, 1600, None, 1, 512, True), (4096, 14336, 704, None, 1, 512, True),
    (8192, 28672, 1600, None, 1, 512, True), (300, 28672, 1600, None, 1, 512, True),
    (64, 49152, 1600, None, 1, 512, True), (40, 8192, 1600, None, 1, 512, True), (1, 16384, 1600, None, 1, 512, True)])
def test_row_segments_are_hardly_larger_than_those_cut_at_tiles(rows, cols, elements, chunk, books, slots, whole):
    """With a row plan, no segment has over 24576 elements and a tenth more
    than the largest of nz_plan_work's, and there are no more of them than run at once; what would
    break that has none (and takes two launches)."""
    elements = elements // 64 * 64
    descs, tiles = plain_tiles(rows, cols, elements, chunk, books)
    row_index, entries = _native.matvec_plan(descs, tiles, [(0, rows)], cols, 2)
    sizes = tiles["n_out"].astype(int)
    for first_weight in (1.0, 1.75):
        segments, _ = _native.matvec_row_plan(descs, tiles, row_index, entries, cols, slots, first_weight)
        cut = _native.plan_work(descs, tiles, slots, first_weight)
        assert bool(len(segments)) == whole
        if whole:
            largest = max(sizes[s["tile0"]:s["tile1"]].sum() for s in cut)
            most = (segments["row1"] - segments["row0"]).astype(int).max() * cols
            assert most <= max(largest + 24576, largest / 0.9)
            assert len(segments) <= max(slots, len(cut))


def run_rows(base, descs, tiles, dtype, weights, cols, x, biases, slots, first_weight):
    """The one-launch form's outputs, whose buffers start as NaN words."""
    spec, batch = DTYPES[dtype], x.shape[0]
    es, reorder = spec.element_size, int(spec.bit_reorder)
    row_index, entries = _native.matvec_plan(descs, tiles, weights, cols, es)
    segments, words = _native.matvec_row_plan(descs, tiles, row_index, entries, cols, slots, first_weight)
    need = words[min(batch - 1, 2)]
    assert len(segments) and need <= _native.lib().nz_matvec_row_words(es, batch)
    records = _native.matvec_tiles(descs, tiles, weights, cols, es, base.size)
    device = [torch.from_numpy(a.view(np.uint8).copy()).cuda() for a in (base, descs, records, row_index)]
    ys = [torch.full((batch * rows * es,), 0xFF, dtype=torch.uint8, device="cuda").view(dtype).view(batch, rows)
          for _, rows in weights]
    xd, bd = x.cuda(), [None if b is None else b.cuda() for b in biases]
    array = _native.matvec_weights([(o, r, y.data_ptr(), None if b is None else b.data_ptr())
                                    for (o, r), y, b in zip(weights, ys, bd)])
    is_long = segments["kind"] == _native.KIND_LONG
    for long_codes, group in enumerate((segments[~is_long], segments[is_long])):
        if len(group):
            part = torch.from_numpy(group.view(np.uint8).copy()).cuda()
            _native.check(_native.lib().nz_matvec_rows(
                device[0].data_ptr(), device[1].data_ptr(), device[2].data_ptr(), part.data_ptr(), len(group), need,
                es, reorder, long_codes, array, len(weights), cols, xd.data_ptr(), batch, device[3].data_ptr(),
                torch.cuda.current_stream().cuda_stream))
            torch.cuda.synchronize()
    return [y.cpu() for y in ys]


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("name", CASES)
def test_one_launch_gives_the_bits_of_two(name, dtype, batch):
    if name == "long" and dtype != torch.bfloat16:
        pytest.skip("the long-code weight is bfloat16")
    base, descs, tiles, weights, cols = case_of(name, dtype)
    g = torch.Generator().manual_seed(batch)
    x = torch.randn(batch, cols, generator=g).to(dtype)
    biases = [(torch.randn(r, generator=g) * 0.1).to(dtype) if i % 2 == 0 else None
              for i, (_, r) in enumerate(weights)]
    (want,) = run_matvec(base, descs, tiles, dtype, weights, cols, x, biases, calls=1)
    for slots, first_weight in ((64, 1.0), (16, 1.75)):
        got = run_rows(base, descs, tiles, dtype, weights, cols, x, biases, slots, first_weight)
        for k, (a, b) in enumerate(zip(got, want)):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), f"weight {k}, {slots} slots"


@pytest.mark.gpu
@pytest.mark.parametrize("dropped", [1, 7, 36, 37])
def test_rows_past_the_weights_are_left_alone(dropped):
    """Row segments of a larger product than the weights say: rows past
    theirs (here still inside the output) keep what they held."""
    base, descs, tiles, weights, cols = case_of("odd-rows", torch.bfloat16)
    rows = weights[0][1] - dropped
    row_index, entries = _native.matvec_plan(descs, tiles, weights, cols, 2)
    segments, words = _native.matvec_row_plan(descs, tiles, row_index, entries, cols, 64)
    records = _native.matvec_tiles(descs, tiles, weights, cols, 2, base.size)
    dev = [torch.from_numpy(a.view(np.uint8).copy()).cuda() for a in (base, descs, records, segments, row_index)]
    x = torch.randn(1, cols, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).cuda()

    def product(named):
        y = torch.full((sum(r for _, r in weights),), float("nan"), dtype=torch.bfloat16, device="cuda")
        array = _native.matvec_weights([(0, named, y.data_ptr(), None)])
        _native.check(_native.lib().nz_matvec_rows(
            *(d.data_ptr() for d in dev[:4]), len(segments), words[0], 2, 1, 0, array, 1, cols, x.data_ptr(), 1,
            dev[4].data_ptr(), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        return y.cpu()

    whole, part = product(sum(r for _, r in weights)), product(rows)
    assert torch.isfinite(whole.float()).all() and torch.isnan(part[rows:].float()).all()
    assert torch.equal(part[:rows].view(torch.int16), whole[:rows].view(torch.int16))


def test_row_launch_refuses_segments_larger_than_the_lds():
    words = _native.lib().nz_matvec_row_words(2, 1)
    assert 1000 < words < 40960
    array = _native.matvec_weights([(0, 1, 1, None)])
    rc = _native.lib().nz_matvec_rows(1, 1, 1, 1, 1, words + 1, 2, 1, 0, array, 1, 2048, 1, 1, 1, None)
    with pytest.raises(_native.NativeError, match="LDS"):
        _native.check(rc)
