"""The primary table's escape entries (codes longer than 12 bits): every one
must lead to the code a window starts with, the kernels' way, as the codes
themselves say."""
import numpy as np
import pytest
import torch

import oracle
from neuralzip_amd import _native
from nz_helpers import Encoded, segment_lengths, segment_tensor

VOCAB = bytes((127, 127, 125, 126))
PRIMARY, SEARCH = 4, 0     # first primary entry; word 0 of an entry that searches the records


def spread_lengths(short, long, top):
    """Complete code over 258 tokens: `short` codes of 1, 2, ... bits, then
    2^k codes each of longer and longer lengths up to `top` bits, so that
    escape prefixes of one length and of several both occur."""
    lengths, room = list(range(1, short + 1)), 1 << (top - short)   # codes of `top` bits left
    for bits in range(13, top):
        take = min(long, room >> (top - bits), 258 - len(lengths))
        while take and (room - (take << (top - bits))) < 258 - len(lengths) - take:
            take -= 1
        lengths += [bits] * take
        room -= take << (top - bits)
    missing = 258 - len(lengths)     # the rest: top bits, the first of them shortened until the code is complete
    lengths += [top] * missing
    spare = room - missing
    for i in range(len(lengths) - 1, -1, -1):
        while spare and lengths[i] > 13 and (1 << (top - lengths[i])) <= spare:
            spare -= 1 << (top - lengths[i])
            lengths[i] -= 1
    assert spare == 0
    return bytes(lengths)


def books():
    counts = [1 << (i // 8) for i in range(258)]
    yield "segment-16", _native.Codebook(b"NZM1" + segment_lengths(16), VOCAB)
    yield "segment-32", _native.Codebook(b"NZM1" + segment_lengths(32), VOCAB)
    yield "segment-33", _native.Codebook(b"NZM1" + segment_lengths(33), VOCAB)
    yield "segment-56", _native.Codebook(b"NZM1" + segment_lengths(56), VOCAB)
    yield "skewed", _native.Codebook(oracle.build_mixed_codebook(counts, VOCAB), VOCAB)
    for short, long, top in ((6, 9, 20), (8, 3, 24)):
        yield f"spread-{short}-{long}-{top}", _native.Codebook(b"NZM1" + spread_lengths(short, long, top), VOCAB)


BOOKS = dict(books())


def entry_token(lut, window):
    """(word of the token, code length) the kernels take for a 64-bit window
    whose primary entry is an escape."""
    x = window >> 52
    e0, e1 = int(lut[PRIMARY + 2 * x]), int(lut[PRIMARY + 2 * x + 1])
    if e0 != SEARCH:
        rest, n = (window >> 20) & 0xFFFFF000, e0 >> 10     # the 20 bits past the prefix, left-justified
        first, second = e0 & 31, e0 >> 5 & 31
        if rest >> first < n:
            return e1 + (rest >> first), 44 - first
        return e1 + n + (rest >> second) - (n << (first - second)), 44 - second
    n, records = int(lut[0]), lut[PRIMARY + 8192:].astype(np.uint64)
    k = e1
    while k + 1 < n and window >= int(records[6 * k]) | int(records[6 * k + 1]) << 32:
        k += 1
    first, length = int(records[6 * k + 2]) | int(records[6 * k + 3]) << 32, int(records[6 * k + 5])
    return PRIMARY + 8192 + 6 * n + int(records[6 * k + 4]) + ((window - first) >> (64 - length)), length


@pytest.mark.parametrize("name", sorted(BOOKS))
def test_every_escape_entry_leads_to_its_code(name):
    book = BOOKS[name]
    lut = book.lut()
    lengths, codes = book.export()
    rng = np.random.default_rng(3)
    escapes = [t for t, n in enumerate(lengths) if n > 12]
    assert escapes
    for t in escapes:
        n, code = int(lengths[t]), int(codes[t])
        width, value = (1, t) if t < 256 else (2, int.from_bytes(VOCAB[2 * (t - 256):2 * (t - 256) + 2], "little"))
        for tail in (0, (1 << (64 - n)) - 1, int(rng.integers(0, 1 << 62)) & ((1 << (64 - n)) - 1)):
            window = (code << (64 - n)) | tail
            assert lut[PRIMARY + 2 * (window >> 52)] >> 27 == 0
            word, length = entry_token(lut, window)
            assert length == n and lut[word] == value | width << 27
    if name == "spread-6-9-20":   # prefixes of one length, of two, and of more
        entries = [int(lut[PRIMARY + 2 * x]) for x in range(4096) if lut[PRIMARY + 2 * x] >> 27 == 0]
        assert {"search" if e == SEARCH else e >> 10 < 0xFFFF for e in entries} == {"search", True, False}


@pytest.mark.parametrize("planted", ["lengths in falling order", "a shift of the whole word", "tokens moved"])
def test_an_escape_entry_that_leads_elsewhere_raises(planted):
    """A mistake planted in the entries of prefixes with two lengths must be
    caught by the emulator's step, whatever the words say."""
    book = BOOKS["spread-6-9-20"]
    symbols = np.random.default_rng(4).permutation(np.repeat(np.arange(256), 20)).astype(np.uint8)
    raw = segment_tensor(torch.bfloat16, symbols)
    base, descs, tiles = Encoded([(raw, torch.bfloat16, 1 << 20, [0], 0)], {0: book}).host_image()
    segments = _native.plan_work(descs, tiles, 4)
    out = np.zeros(raw.size + 64, dtype=np.uint8)
    _native.emulate_decode(base, descs, tiles, segments, 2, 1, out)
    assert np.array_equal(out[:raw.size], raw)
    image = base[int(descs["lut"][0]):].view(np.uint32)
    two = [PRIMARY + 2 * x for x in range(4096) if image[PRIMARY + 2 * x] >> 27 == 0 and image[PRIMARY + 2 * x] != SEARCH
           and image[PRIMARY + 2 * x] >> 10 < 0xFFFF]
    assert two
    for at in two:
        first, second, n = int(image[at]) & 31, int(image[at]) >> 5 & 31, int(image[at]) >> 10
        image[at] = {"lengths in falling order": second | first << 5 | n << 10,
                     "a shift of the whole word": 0 | second << 5 | n << 10,
                     "tokens moved": int(image[at])}[planted]
        image[at + 1] += planted == "tokens moved"
    with pytest.raises(_native.NativeError, match="Escape entry does not lead"):
        _native.emulate_decode(base, descs, tiles, segments, 2, 1, out)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("name", sorted(BOOKS))
def test_escape_heavy_tiles_decode(name, dtype):
    """Every code equally often beside runs of the shortest ones: escapes in
    all lanes of a step, in a few and in none, against the original words
    and the CPU emulation."""
    from test_gpu_decode import check_case
    rng = np.random.default_rng(9)
    symbols = np.concatenate([rng.permutation(np.repeat(np.arange(256), 20)),
                              np.where(rng.random(30000) < 0.02, rng.integers(0, 256, 30000), 127),
                              np.full(3001, 127)]).astype(np.uint8)
    raw = segment_tensor(dtype, symbols)
    check_case([(raw, dtype, 16384, [0] * -(-symbols.size // 16384), 37)], {0: BOOKS[name]}, dtype)
