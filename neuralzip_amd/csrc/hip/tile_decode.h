// tile_decode.h -- wave64 tile decode shared by the gfx950 kernels.
//
// Device code only. A wavefront decodes one tile of the layout in
// nz_format.h into its LDS staging area (one exponent byte per element);
// the kernels differ in what they do with the staged bytes: the decode
// kernel merges them with the raw lanes and stores the words, the
// matrix-vector kernel multiplies the merged words by an activation vector.
#ifndef NZ_TILE_DECODE_H
#define NZ_TILE_DECODE_H

#include <hip/hip_runtime.h>

#include <stdint.h>

#include "../nz_format.h"

namespace {

constexpr int kIcmpUge = 35, kIcmpUlt = 36;   // unsigned predicates of the lane-mask compare builtin
// s_waitcnt operand (gfx9 encoding) that waits for every outstanding LDS
// operation: lgkmcnt 0, vmcnt 63 and expcnt 7 (no wait on those).
constexpr int kWaitLgkm0 = 0xC07F;

__device__ __forceinline__ uint32_t bswap32(uint32_t x) { return __builtin_amdgcn_perm(0u, x, 0x00010203u); }

__device__ __forceinline__ uint32_t funnel(uint32_t hi, uint32_t lo, uint32_t s) {
    return __builtin_amdgcn_alignbit(hi, lo, s);
}

// Bit-field insert: bits of `a` where `mask` is set, bits of `b` elsewhere.
__device__ __forceinline__ uint32_t bfi(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | (b & ~mask); }

// Buffer resources: a wave-uniform base and byte range; loads outside the
// range return zero and stores outside it are dropped, so every lane issues
// the same memory instructions whether or not its element exists. Word 3
// selects 32-bit raw data, the untyped layout of the gfx9 family.
constexpr uint32_t kRawBufferFlags = 0x00020000u;
constexpr uint32_t kOutOfRange = 0x80000000u;
// Cache-policy operand of buffer stores: streaming (nontemporal) writes of
// the decoded words, which the caches need not keep.
constexpr int kNonTemporal = 2;
using rsrc_t = __amdgpu_buffer_rsrc_t;
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

__device__ __forceinline__ rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, kRawBufferFlags);
}

// Inclusive prefix sum over the wavefront: shifts of 1, 2, 4, 8 lanes inside
// each row of 16, then the row carries (row_bcast:15 into rows 1 and 3,
// row_bcast:31 into rows 2 and 3).
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x111, 0xF, 0xF, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x112, 0xF, 0xF, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x114, 0xF, 0xF, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x118, 0xF, 0xF, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x142, 0xA, 0xF, false));
    v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x143, 0xC, 0xF, false));
    return v;
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Canonical decode of one code longer than 12 bits whose prefix holds codes
// of three or more lengths, or longer than 32 bits: from record `k` on, find
// the first escape length whose left-justified limit exceeds the window.
// Returns the image word of the code's token; *len receives its length.
// Without LONG all codes end within the window's first 32 bits.
template <bool LONG>
__device__ __forceinline__ uint32_t escape_search(const uint32_t* lut, uint32_t w0, uint32_t w1, uint32_t k,
                                                  uint32_t* len) {
    const uint32_t records = NZ_LUT_HEADER + 2 * NZ_LUT_ENTRIES, tokens = records + NZ_ESC_RECORD * lut[0];
    uint32_t r = records + NZ_ESC_RECORD * k;
    const uint64_t window = (static_cast<uint64_t>(w0) << 32) | w1;
    for (; r + NZ_ESC_RECORD < tokens; r += NZ_ESC_RECORD)
        if (LONG ? window < (lut[r] | (static_cast<uint64_t>(lut[r + 1]) << 32)) : w0 < lut[r + 1]) break;
    const uint32_t L = lut[r + 5];
    *len = L;
    const uint32_t offset =
        LONG ? static_cast<uint32_t>((window - (lut[r + 2] | (static_cast<uint64_t>(lut[r + 3]) << 32))) >> (64 - L))
             : (w0 - lut[r + 3]) >> (32 - L);
    return tokens + lut[r + 4] + offset;
}

template <int ES, bool REORDER>
__device__ __forceinline__ uint32_t restore_word(uint32_t v) {
    if (!REORDER) return v;
    if (ES == 2)   // two bfloat16 per dword
        return (v & 0x007F007Fu) | ((v << 8) & 0x80008000u) | ((v >> 1) & 0x7F807F80u);
    return (v & 0x007FFFFFu) | ((v << 8) & 0x80000000u) | ((v >> 1) & 0x7F800000u);
}

// Staged form of exponent bytes: with REORDER each byte is rotated right by
// one bit, so that exponent >> 1 and the exponent's lowest bit sit where the
// restored bytes hold them and merging takes one bit-field insert per dword
// instead of a shift and an insert (8 of a 16-byte vector's 20 vector
// instructions before). The LUT's copy in LDS holds its bytes in this form.
template <bool REORDER>
__device__ __forceinline__ uint32_t staged_form(uint32_t e) {
    return REORDER ? bfi(0x7F7F7F7Fu, e >> 1, e << 7) : e;
}

// One element's word from its staged exponent byte and its raw lane bytes
// `raw` (lane k in byte k).
template <int ES, bool REORDER>
__device__ __forceinline__ uint32_t element_word(uint32_t staged, uint32_t raw) {
    const uint32_t expo = REORDER ? ((staged << 1) | (staged >> 7)) & 0xFFu : staged;
    return restore_word<ES, REORDER>((expo << (8 * (ES - 1))) | raw);
}

// Four elements' top two bytes from four staged exponent bytes `e` and the
// four stored bytes below them `r` (bit 7 = sign when reordered): returns the
// restored high bytes in *hi and the bytes below them in *lo.
template <bool REORDER>
__device__ __forceinline__ void restore_pairs(uint32_t e, uint32_t r, uint32_t* hi, uint32_t* lo) {
    if (REORDER) {
        *hi = bfi(0x7F7F7F7Fu, e, r);    // sign | exponent >> 1
        *lo = bfi(0x7F7F7F7Fu, r, e);    // exponent bit 0 | low mantissa bits
    } else {
        *hi = e;
        *lo = r;
    }
}

// A whole 16-byte vector of V elements. `e` holds V staged exponent bytes (two
// dwords for 2-byte words, one for 4-byte words); `r` the raw lane dwords
// (lane 0 for 2-byte words; lanes 0, 1, 2 for 4-byte words).
template <int ES, bool REORDER>
__device__ __forceinline__ uint4 merge_vector(uint32_t e0, uint32_t e1, const uint32_t* r) {
    uint4 v;
    if (ES == 2) {
        uint32_t hi, lo;
        restore_pairs<REORDER>(e0, r[0], &hi, &lo);
        v.x = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
        v.y = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
        restore_pairs<REORDER>(e1, r[1], &hi, &lo);
        v.z = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
        v.w = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
    } else {
        uint32_t hi, lo;
        restore_pairs<REORDER>(e0, r[2], &hi, &lo);
        const uint32_t a = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);
        const uint32_t b = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
        const uint32_t c = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
        const uint32_t d = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
        v.x = __builtin_amdgcn_perm(c, a, 0x05040100u);
        v.y = __builtin_amdgcn_perm(c, a, 0x07060302u);
        v.z = __builtin_amdgcn_perm(d, b, 0x05040100u);
        v.w = __builtin_amdgcn_perm(d, b, 0x07060302u);
    }
    return v;
}


template <int ES>
struct Geometry {
    static constexpr uint32_t V = 16 / ES;                        // elements per 16-byte vector
    static constexpr uint32_t kCapacity = ES == 4 ? NZ_TILE_OUT32 : NZ_TILE_OUT;
    static constexpr uint32_t kStage = NZ_STAGE_ORIGIN + kCapacity + NZ_STAGE_SLACK;
    // a tile's vectors (its first element's offset in its vector included)
    // never exceed the capacity
    static constexpr uint32_t kRounds = kCapacity / V / NZ_WAVE;
    static constexpr uint32_t kLaneWords = ES == 2 ? 2 : 3;       // raw-lane dwords per vector
};

// Wave-uniform description of one tile (scalar registers).
struct TileInfo {
    const uint8_t* bits;       // first window of the tile
    const uint16_t* meta;      // its metadata
    const uint8_t* lanes;      // raw lane 0 at the tile's first vector
    uint64_t first;            // workspace element at staging index 0 (a multiple of V)
    uint32_t stride;           // raw lane stride
    uint32_t n_win;
    uint32_t skip;             // bytes of the first window that belong to the previous tile
    uint32_t s0, s1;           // staging indices of the first and one-past-last element
    uint32_t nv;               // vectors covering [s0, s1)
};

template <int ES>
__device__ __forceinline__ TileInfo tile_info(const uint8_t* base, const nz_frag_desc* frags, const nz_tile* tiles,
                                              uint32_t t) {
    constexpr uint32_t V = Geometry<ES>::V;
    const nz_tile tile = tiles[t];
    const nz_frag_desc f = frags[tile.frag];
    const uint64_t a0 = f.out + tile.out0;
    const uint64_t vbase = a0 / V;
    const uint64_t origin = f.out / V * V;
    TileInfo ti;
    ti.bits = base + f.bits + 8ull * tile.win0;
    ti.meta = reinterpret_cast<const uint16_t*>(base + f.meta) + tile.win0;
    ti.lanes = base + f.lanes + (vbase * V - origin);
    ti.first = vbase * V;
    ti.stride = f.lane_stride;
    ti.n_win = nz_tile_windows(tile.counts);
    ti.skip = nz_tile_skip(tile.counts);
    ti.s0 = static_cast<uint32_t>(a0 - vbase * V);
    ti.s1 = ti.s0 + nz_tile_elements(tile.counts);
    ti.nv = (ti.s1 + V - 1) / V;
    return ti;
}

// Staging index of the edge element lane `lane` owns in the edge round:
// lanes [0, V) the first vector, lanes [V, 2V) the last one.
template <int ES>
__device__ __forceinline__ uint32_t edge_index(const TileInfo& ti, uint32_t lane) {
    constexpr uint32_t V = Geometry<ES>::V;
    return lane < V ? lane : (ti.nv - 1) * V + (lane & (V - 1));
}


// Everything a lane reads from global memory for one tile. All loads are
// unconditional with clamped indices, so the compiler's wait counts stay
// exact while the next tile's loads are in flight.
template <int ES, bool LONG>
struct Fetch {
    uint32_t meta;
    uint32_t w[LONG ? 4 : 3];
    uint32_t raw[Geometry<ES>::kRounds][Geometry<ES>::kLaneWords];
};

// The part of a tile's data the decode needs first: window metadata and bits.
template <int ES, bool LONG>
__device__ __forceinline__ void fetch_bits(const TileInfo& ti, uint32_t lane, Fetch<ES, LONG>& d) {
    const rsrc_t meta = make_rsrc(ti.meta, 2 * ti.n_win);
    const rsrc_t bits = make_rsrc(ti.bits, 8 * ti.n_win + NZ_BITS_PAD);
    d.meta = __builtin_amdgcn_raw_buffer_load_b16(meta, 2 * lane, 0, 0);
    {   // the lane's window and the 64 bits after it
        const v4u w = __builtin_amdgcn_raw_buffer_load_b128(bits, 8 * lane, 0, 0);
        d.w[0] = w.x;
        d.w[1] = w.y;
        d.w[2] = w.z;
        if (LONG) d.w[3] = w.w;
    }
}

// Merge rounds that a tile of 16-bit words may not reach: 64 windows hold
// anything from a few hundred elements (fp16: about 740) to the limit. The
// fused kernel leaves their loads out by scalar branches: 4096 x 14336 fp16
// took 41.9 us with the loads of all rounds in every tile and 32.8 without,
// for four activation rows 71.7 and 56.1; 28672 x 4096 bf16 (tiles of 1600,
// all four rounds) 43.8 and 43.0. 32-bit words reach their limit but with
// codes over four bits, and the branches alone cost them 2 %.
template <int ES>
constexpr bool late_round(uint32_t r) { return ES == 2 && r >= 2; }

// The part used only after the decode: raw lanes. With TRIM, rounds that the
// tile does not reach (late_round) are left out by a scalar branch.
template <int ES, bool LONG, bool TRIM = false>
__device__ __forceinline__ void fetch_raw(const TileInfo& ti, uint32_t lane, Fetch<ES, LONG>& d) {
    using G = Geometry<ES>;
    const uint32_t span = ti.nv * G::V;   // lane bytes covering the tile's vectors
    const rsrc_t lanes = make_rsrc(ti.lanes, ES == 2 ? span : 2 * ti.stride + span);
#pragma unroll
    for (uint32_t r = 0; r < G::kRounds; ++r) {
        if (TRIM && late_round<ES>(r) && ti.s1 <= r * NZ_WAVE * G::V) break;
        const uint32_t at = (lane + NZ_WAVE * r) * G::V;
        if (ES == 2) {
            const v2u v = __builtin_amdgcn_raw_buffer_load_b64(lanes, at, 0, 0);
            d.raw[r][0] = v.x;
            d.raw[r][1] = v.y;
        } else {
            d.raw[r][0] = __builtin_amdgcn_raw_buffer_load_b32(lanes, at, 0, 0);
            d.raw[r][1] = __builtin_amdgcn_raw_buffer_load_b32(lanes, at + ti.stride, 0, 0);
            d.raw[r][2] = __builtin_amdgcn_raw_buffer_load_b32(lanes, at + 2 * ti.stride, 0, 0);
        }
    }
}

// Raw lane bytes (lane k in byte k) of the element at staging index g of one
// of a tile's partial vectors, 0 for a lane without one (kOutOfRange). Tiles
// end on whole vectors but at a fragment's unaligned ends, so the load is
// left to the tiles that have such elements.
template <int ES>
__device__ __forceinline__ uint32_t edge_raw(const TileInfo& ti, uint32_t g) {
    const uint32_t span = ti.nv * Geometry<ES>::V;
    const rsrc_t lanes = make_rsrc(ti.lanes, ES == 2 ? span : 2 * ti.stride + span);
    uint32_t raw = __builtin_amdgcn_raw_buffer_load_b8(lanes, g, 0, 0);
    if (ES == 4)
        raw |= (static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b8(lanes, g + ti.stride, 0, 0)) << 8) |
               (static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b8(lanes, g + 2 * ti.stride, 0, 0)) << 16);
    return raw;
}

__device__ __forceinline__ uint2 lut_entry(const uint32_t* lut, uint32_t w0) {
    return reinterpret_cast<const uint2*>(lut + NZ_LUT_HEADER)[w0 >> (32 - NZ_LUT_BITS)];
}

// One LUT step at the head of the window w0..w3, whose primary entry is `e`:
// returns the step's entry (byte count in bits 27-29 of .x; the bytes, first
// lowest and zeros above them, in .y) and shifts the window by the consumed
// bits.
template <bool LONG, bool ESC>
__device__ __forceinline__ uint2 lut_step(const uint32_t* lut, uint2 e, uint32_t& w0, uint32_t& w1, uint32_t& w2,
                                          uint32_t& w3) {
    if (ESC) {
        // One scalar branch where no lane escapes (0.8 % of a lane's steps
        // do, so three steps in ten of a wavefront), and inside it one more
        // where all lanes' codes have their prefix's first length; the empty
        // asm keeps the compiler from folding the lanes' tests into them. An
        // escape entry names the token of almost every escape, one LDS read:
        // searching the length records for each one took 35 % of the fused
        // kernel's vector instructions and 65 % of its scalar ones.
        if (__builtin_expect(__builtin_amdgcn_uicmp(e.x, 1u << NZ_ENTRY_COUNT, kIcmpUlt) != 0, 0)) {
            asm volatile("");
            if (e.x < (1u << NZ_ENTRY_COUNT)) {
                // codes of one length under the prefix count up from its first token
                const uint32_t rest = w0 << NZ_LUT_BITS, n = e.x >> NZ_ESC_COUNT;
                uint32_t token = e.y + (rest >> (e.x & 31u)), s = e.x - NZ_LUT_BITS;
                if (__builtin_expect(__builtin_amdgcn_uicmp(rest >> (e.x & 31u), n, kIcmpUge) != 0, 0)) {
                    asm volatile("");
                    if (e.x == NZ_ESC_SEARCH) {
                        uint32_t len;
                        token = escape_search<LONG>(lut, w0, w1, e.y, &len);
                        if (LONG && len > 32) {
                            w0 = w1;
                            w1 = w2;
                            w2 = w3;
                            w3 = 0;
                            len -= 32;
                        }
                        s = 32 - len;   // len in [1, 32]; s == 0 shifts a whole word
                    } else if (rest >> (e.x & 31u) >= n) {   // the prefix's second length
                        s = (e.x >> NZ_ESC_SECOND) & 31u;
                        token = e.y + n + (rest >> s) - (n << ((e.x & 31u) - s));
                        s -= NZ_LUT_BITS;
                    }
                }
                const uint32_t t = lut[token];
                e.y = t & 0xFFFFu;   // one or two bytes
                e.x = bfi(31u, s, t & ~0xFFFFu);
            }
        }
    }
    // the funnel shift reads its low five bits
    w0 = funnel(w0, w1, e.x);
    w1 = funnel(w1, w2, e.x);
    w2 = funnel(w2, LONG ? w3 : 0u, e.x);
    if (LONG) w3 = funnel(w3, 0u, e.x);
    return e;
}

// A lane's place in a tile's decode: its window, left-justified at the next
// code, and its place in the staging area as -8 x the LDS byte address of its
// next byte (`neg`) and of the byte after its last one (`stop`).
struct LaneDecode {
    uint32_t w0, w1, w2, w3;
    uint32_t neg, stop;
};

// Clears the tile's staging bytes and sets up the decode of a tile from
// its metadata and windows in `d`, which are free for the next tile after it.
template <int ES, bool LONG>
__device__ __forceinline__ LaneDecode open_tile(const TileInfo& ti, const Fetch<ES, LONG>& d, uint8_t* stage,
                                                uint32_t lane) {
    using G = Geometry<ES>;
    // what the merge reads: the rounds that hold elements of the tile
#pragma unroll
    for (uint32_t r = 0; r < G::kCapacity / (8 * NZ_WAVE); ++r)
        if (r < 2 || ti.s1 > 2 * 8 * NZ_WAVE)
            *reinterpret_cast<uint2*>(stage + NZ_STAGE_ORIGIN + 8 * (lane + NZ_WAVE * r)) = make_uint2(0u, 0u);
    const uint32_t count = d.meta >> 8;   // 0 past the tile's windows: their metadata loads are out of range
    // The first window's skipped bytes land in the staging area's prefix
    // (NZ_STAGE_ORIGIN exceeds any skip, so the address stays inside it).
    const uint32_t base = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)stage));
    const uint32_t end = base + NZ_STAGE_ORIGIN + ti.s0 - ti.skip + wave_inclusive_scan(count);
    LaneDecode l;
    l.stop = 0u - 8u * end;
    l.neg = l.stop + 8u * count;
    l.w0 = bswap32(d.w[0]), l.w1 = bswap32(d.w[1]), l.w2 = bswap32(d.w[2]), l.w3 = LONG ? bswap32(d.w[3]) : 0u;
    uint32_t g = d.meta & 0xFFu;   // restart at the gap
    if (LONG) {
        if (g >= 32) { l.w0 = l.w1; l.w1 = l.w2; l.w2 = l.w3; l.w3 = 0; g -= 32; }
        if (g) {
            const uint32_t s = 32 - g;
            l.w0 = funnel(l.w0, l.w1, s);
            l.w1 = funnel(l.w1, l.w2, s);
            l.w2 = funnel(l.w2, l.w3, s);
            l.w3 = funnel(l.w3, 0u, s);
        }
    } else {   // codes end within the window's 95 bits, so the gap is at most 31
        const uint64_t high = ((static_cast<uint64_t>(l.w0) << 32) | l.w1) << g;
        const uint64_t low = ((static_cast<uint64_t>(l.w1) << 32) | l.w2) << g;
        l.w0 = static_cast<uint32_t>(high >> 32);
        l.w1 = static_cast<uint32_t>(low >> 32);
        l.w2 = static_cast<uint32_t>(low);
    }
    return l;
}

// Decodes a tile's exponent bytes into the wavefront's cleared staging area:
// staging index i (from NZ_STAGE_ORIGIN) holds the staged exponent byte of the
// element at workspace index ti.first + i, for i in [ti.s0, ti.s1). Ends with
// the wavefront's LDS writes visible to all of its lanes.
//
// Every write into the area is an LDS atomic OR of whole aligned
// dwords, so lanes may share a dword without any ordering between them. A
// lane's bytes go to [neg, stop); its final LUT step may emit up to three
// bytes past them, and those are the next window's first bytes (the bitstream
// is continuous: decoding on past a window's last code decodes the codes that
// start in the next window), or, after the tile's last window, bytes that no
// one reads. An OR therefore only ever adds a byte's own value or zeros.
template <bool LONG, bool ESC>
__device__ __forceinline__ void decode_tile(LaneDecode l, const uint32_t* lut) {
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    if (l.neg > l.stop) {
        uint2 e = lut_entry(lut, l.w0);
        do {
            e = lut_step<LONG, ESC>(lut, e, l.w0, l.w1, l.w2, l.w3);
            // The entry's bytes go to [p, p + count): the dword of byte
            // p - 1 and the one after it, so that two funnel shifts by
            // 32 - 8 (p mod 4), zero for an aligned p, split them.
            lds_u32* dst = (lds_u32*)(uintptr_t)static_cast<uint32_t>(~((static_cast<int32_t>(l.neg) >> 3) | 3));
            const uint32_t low = funnel(e.y, 0u, l.neg), high = funnel(0u, e.y, l.neg);
            l.neg -= e.x >> (NZ_ENTRY_COUNT - 3);   // 8 x the byte count (bits 26 and 25 of a step's entry are zero)
            // The next step's LUT read is issued before this step's ORs, so
            // that their latencies overlap; the last one's entry goes
            // unused. Nothing is left for a register copy: all uses of the
            // entry come before the read that replaces it.
            __builtin_amdgcn_sched_barrier(0);
            e = lut_entry(lut, l.w0);
            __hip_atomic_fetch_or(dst, low, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            __hip_atomic_fetch_or(dst + 1, high, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            // The read and the ORs complete before the wavefront issues its
            // next LDS instruction. On gfx950 an LDS read issued while the
            // same wavefront's LDS atomics were still in flight has returned
            // staging data in place of the LUT entry, now and then.
            __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
        } while (l.neg > l.stop);
    }
    wave_lds_sync();
}

// A segment's LUT image on its way into LDS: the header and the primary
// entries, whose place and number are the same in every image, are requested
// at once by fetch(); store() writes them in staged form and copies the
// escape records and tokens behind them, whose number the header gives.
// (Reading the size first, then copying in a loop that waits for each of its
// loads, put four memory latencies one after the other ahead of a
// workgroup's first tile; two are left. With the decode kernel's first tiles
// requested beside it, 14.9 M bf16 elements went from 11.0 to 10.7 us of
// kernel time and 13.1 M fp32 elements from 17.8 to 16.9.)
template <bool REORDER, int THREADS>
struct LutCopy {
    static constexpr uint32_t kPrimary = NZ_LUT_ENTRIES / 2;   // 16-byte vectors of two entries
    static constexpr uint32_t kRounds = (kPrimary + THREADS - 1) / THREADS;
    const uint4* image;
    uint4 head;
    uint4 v[kRounds];

    __device__ __forceinline__ void fetch(const uint8_t* at, uint32_t thread) {
        image = reinterpret_cast<const uint4*>(at);
        head = image[0];
#pragma unroll
        for (uint32_t r = 0; r < kRounds; ++r)
            v[r] = image[1 + (kPrimary % THREADS ? min(thread + r * THREADS, kPrimary - 1) : thread + r * THREADS)];
    }

    __device__ __forceinline__ void store(uint32_t* lut, uint32_t thread) {
        uint4* dst = reinterpret_cast<uint4*>(lut);
        // the host checks every image against NZ_LUT_MAX_WORDS; the clamp keeps a
        // malformed one from overwriting the staging areas behind the LUT
        const uint32_t words = min(head.z, uint32_t(NZ_LUT_MAX_WORDS));
        const uint32_t tokens = NZ_LUT_HEADER + 2 * NZ_LUT_ENTRIES + NZ_ESC_RECORD * head.x;
        const uint32_t i = 1 + kPrimary + thread;   // escape records and tokens: 212 vectors at most
        static_assert((NZ_LUT_MAX_WORDS + 3) / 4 - 1 - kPrimary <= THREADS, "one vector per thread");
        const bool tail = i < (words + 3) / 4;
        uint4 e = make_uint4(0u, 0u, 0u, 0u);
        if (tail) e = image[i];
        if (thread == 0) dst[0] = head;
#pragma unroll
        for (uint32_t r = 0; r < kRounds; ++r) {
            if (kPrimary % THREADS != 0 && thread + r * THREADS >= kPrimary) break;
            if (v[r].x >> NZ_ENTRY_COUNT) v[r].y = staged_form<REORDER>(v[r].y);
            if (v[r].z >> NZ_ENTRY_COUNT) v[r].w = staged_form<REORDER>(v[r].w);
            dst[1 + thread + r * THREADS] = v[r];
        }
        if (tail) {
            if (REORDER) {   // escape tokens: two bytes below the count
                uint32_t* w = &e.x;
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k)
                    if (4 * i + k >= tokens) w[k] = bfi(0xFFFFu, staged_form<true>(w[k] & 0xFFFFu), w[k]);
            }
            dst[i] = e;
        }
    }
};

// A workgroup's LDS. The claim counter comes first: ds_append takes its
// address from M0's low 16 bits, which reach the first 64 KB.
template <int ES, int WAVES>
struct GroupLds {
    uint32_t claim[4];
    uint32_t lut[(NZ_LUT_MAX_WORDS + 3) / 4 * 4];
    uint8_t stage[WAVES][Geometry<ES>::kStage];
};

// This thread's lane. The compiler does not see its range, so it keeps
// lane * size + constant as an address and an immediate offset instead of one
// register per constant.
__device__ __forceinline__ uint32_t lane_index() {
    uint32_t lane = threadIdx.x % NZ_WAVE;
    asm("" : "+v"(lane));
    return lane;
}

// The next tile index of the workgroup's segment for this wavefront: one
// ds_append, which adds the number of its active lanes (all 64) to the
// counter. Indices at or past the segment's size mean it is used up.
__device__ __forceinline__ uint32_t claim(uint32_t* counter) {
    typedef __attribute__((address_space(3))) int lds_int;
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(__builtin_amdgcn_ds_append((lds_int*)counter))) / NZ_WAVE;
}

}  // namespace

#endif
