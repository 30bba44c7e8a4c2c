// Rows of the expert formats, decoded a quarter block (64 of 256 columns) per lane into eight signed, scaled fp16 weights at a time: what
// the MFMA kernels on tiles of tokens and on one token share.
#pragma once
#include <type_traits>
#include <utility>

#include "redhip_mfma.h"

namespace redhip {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
union H8 { uint4 u; half8_t v; half2_t p[4]; _Float16 e[8]; };

// row sources: format (low half, what the decode goes by) and layout
enum : int { F_XXS = 0, F_XS = 1, F_M = 2, F_IQ3 = 3, F_IQ3_WORDS = 4, L_RAW = 0, L_ROWS = 8, L_TILED = 16 };
enum : int { S_XXS = F_XXS, S_XS = F_XS, S_M = F_M, S_IQ3 = F_IQ3, S_ROWS_XXS = F_XXS | L_ROWS, S_TILED_XXS = F_XXS | L_TILED, S_TILED_XS = F_XS | L_TILED,
             S_TILED_M = F_M | L_TILED, S_TILED_IQ3 = F_IQ3_WORDS | L_TILED };
// a kernel on one token uses every table entry about once: small tables, quickly built
enum : int { SMALL_TABLES = 32 };
template <int SRC> constexpr bool small_tables() { return (SRC & SMALL_TABLES) != 0; }
template <int SRC> constexpr int fmt() { return SRC & 7; }
template <int SRC> constexpr int layout() { return SRC & 24; }
// bytes per 256 columns of a row: raw blocks; the quarters of the other layouts (their block scales lie apart)
template <int SRC> constexpr uint32_t src_block() {
    return layout<SRC>() != L_RAW ? (fmt<SRC>() == F_IQ3_WORDS ? 128u : 64u) : fmt<SRC>() == F_XXS ? 66u : fmt<SRC>() == F_XS ? 74u : fmt<SRC>() == F_M ? 56u : 110u;
}
template <int SRC> constexpr float format_scale() { return fmt<SRC>() == F_XXS || fmt<SRC>() == F_XS ? 0.125f : 1.0f; }      // the d / 8 of the IQ2 formats
// first of the eight columns that lane quarter q multiplies in step s of a block: its own quarter, in order - or, where the lane reads entry q
// of every group (tile-major IQ3_S words), that entry
template <int SRC> __device__ __forceinline__ uint32_t step_column(uint32_t s, uint32_t q) { return fmt<SRC>() == F_IQ3_WORDS ? 128u * (s >> 2) + 32u * (s & 3u) + 8u * q : 64u * q + 8u * s; }

// Decode tables in LDS.
//   IQ2_XXS: the eight fp16 magnitudes of every grid entry times every group scale 2 s + 1 (64 KB, exact), at entry * 256 + s * 16: the address is
//   the entry's byte over the top byte of the group's second word, one byte permute and one mask; IQ3_S likewise (four magnitudes, by scale)
//   IQ2_XS: the fp16 codebook eight times, lane l reading copy l % 8 - a wave's 16-byte reads then hit every bank evenly (random entries of
//   one copy: 2.6 times the cycles); IQ1_M: its codebook with the offset of +1/8 and of -1/8, at (offset sign << 15 | entry << 4)
//   Small tables (32 KB, IQ3_S 16): IQ2_XXS and IQ3_S without the scales, eight and four copies; IQ2_XS four copies, IQ1_M one
//   signs: bit 15 - i / 31 - i of the word of a sign field = signs of weights 2i and 2i + 1, so a pair's signs are one shift and one and-or;
//   replicated so that the reads are (nearly) free of conflicts. (Sign masks as 16-byte entries save three shifts per eight weights and cost
//   a second conflicting 16-byte read: LDS, the tighter of the two pipes, loses more.)
template <int SRC> constexpr bool is_iq3() { return fmt<SRC>() == F_IQ3 || fmt<SRC>() == F_IQ3_WORDS; }
template <int SRC> constexpr uint32_t sign_copies() { return fmt<SRC>() == F_M ? 0u : small_tables<SRC>() ? (is_iq3<SRC>() ? 2u : 4u) : is_iq3<SRC>() ? 4u : 32u; }
template <int SRC> constexpr uint32_t sign_shift() { return sign_copies<SRC>() == 32u ? 7u : sign_copies<SRC>() == 4u ? 4u : 3u; }
template <int SRC> constexpr uint32_t sign_bytes() { return (is_iq3<SRC>() ? 256u : 128u) * sign_copies<SRC>() * 4u; }
constexpr uint32_t kEntryBytes = 65536u;

template <int SRC> constexpr uint32_t codebook_entries() { return fmt<SRC>() == F_XXS ? 256u : fmt<SRC>() == F_M ? 2048u : 512u; }

// Bytes B and B + 1 of w as two fp16 halves: 1024 + byte by a permute (100 0100 of the exponent above it), minus 1024, exact. Signed bytes: flipped to
// 0 .. 255 before, minus another 128.
template <uint32_t B, bool SIGNED> __device__ __forceinline__ half2_t byte_halves(uint32_t w) {
    const half2_t v = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, SIGNED ? w ^ 0x80808080u : w, 0x04000400u | B | ((B + 1u) << 16)));
    constexpr _Float16 off = SIGNED ? 1152.0f : 1024.0f;
    return v - half2_t{off, off};
}
template <bool SIGNED> __device__ __forceinline__ H8 entry_halves(uint64_t e) {
    H8 r;
    r.p[0] = byte_halves<0u, SIGNED>((uint32_t)e);
    r.p[1] = byte_halves<2u, SIGNED>((uint32_t)e);
    r.p[2] = byte_halves<0u, SIGNED>((uint32_t)(e >> 32));
    r.p[3] = byte_halves<2u, SIGNED>((uint32_t)(e >> 32));
    return r;
}
__device__ __forceinline__ half2_t odd_halves(uint32_t s) {      // 2 s + 1 twice, exact
    const half2_t big = __builtin_bit_cast(half2_t, (0x6401u + 2u * s) * 0x10001u);
    return big - half2_t{(_Float16)1024.0f, (_Float16)1024.0f};
}

template <int SRC, uint32_t T>          // by T threads
__device__ __forceinline__ void build_signs(uint32_t *signs, uint32_t tid) {
    if constexpr (fmt<SRC>() != F_M) {
        constexpr uint32_t R = sign_copies<SRC>(), W = R < 4u ? R : 4u, N = sign_bytes<SRC>() / (4u * W);      // W copies a store
        for (uint32_t i = tid; i < N; i += T) {
            const uint32_t s = i * W / R, s8 = is_iq3<SRC>() ? s : s | ((__popc(s) & 1u) << 7);
            uint32_t y = ((s8 >> 1) & 0x55u) | ((s8 & 0x55u) << 16);      // odd weights' signs in the low half, even ones' in the high half, side by side, then in reverse
            y = (y | (y >> 1)) & 0x00330033u;
            y = (y | (y >> 2)) & 0x000f000fu;
            const uint32_t w = __brev(y);
            if constexpr (W == 4u) reinterpret_cast<uint4 *>(signs)[i] = make_uint4(w, w, w, w);
            else reinterpret_cast<uint2 *>(signs)[i] = make_uint2(w, w);
        }
    }
}

// The large tables, by T threads in two parts: a thread's codebook entries are requested together (a trip to memory, beside whatever is requested behind
// them), then written: every further entry is packed fp16 arithmetic, exact.
// Where a thread writes four entries side by side, in an order that differs between the fours of lanes: sixteen lanes then write to different
// banks. (Entry by entry in f32, each behind a trip of its own, the tables of IQ2_XXS took 8000 cycles of every launch, of the 91000 of a batch
// of 24 tokens.)
template <int SRC, uint32_t T> struct TableSeeds {
    // items: XXS four scales of an entry, XS four copies, M an entry with both offsets, IQ3 eight scales of an entry
    static constexpr uint32_t kPer = fmt<SRC>() == F_XXS ? 4u : fmt<SRC>() == F_M ? 1u : 2u, kItems = kPer * codebook_entries<SRC>(), N = (kItems + T - 1u) / T;
    std::conditional_t<is_iq3<SRC>(), uint32_t, uint64_t> e[N];
    static __device__ __forceinline__ uint32_t item(uint32_t tid, uint32_t n) { return min(tid + n * T, kItems - 1u); }      // (surplus threads repeat the last)
    __device__ __forceinline__ void request(uint32_t tid, const int8_t *grid) {
#pragma unroll
        for (uint32_t n = 0; n < N; ++n) {
            const uint32_t i = item(tid, n);
            if constexpr (is_iq3<SRC>()) e[n] = redhip_iq3s_grid[i & 511u];
            else if constexpr (fmt<SRC>() == F_XXS) e[n] = redhip_iq2xxs_grid[i / kPer];
            else e[n] = reinterpret_cast<const uint64_t *>(grid)[i / kPer];
        }
    }
    __device__ __forceinline__ void store(uint8_t *entries, uint32_t *signs, uint32_t tid) const {
        build_signs<SRC, T>(signs, tid);
#pragma unroll
        for (uint32_t n = 0; n < N; ++n) {
            const uint32_t i = item(tid, n);
            if constexpr (is_iq3<SRC>()) {
                const half2_t a = byte_halves<0u, false>(e[n]), b = byte_halves<2u, false>(e[n]);
#pragma unroll
                for (uint32_t k = 0; k < 8u; ++k) {
                    const uint32_t scale = (i >> 9) * 8u + k;
                    const half2_t f = odd_halves(scale);
                    *reinterpret_cast<uint2 *>(entries + (scale * 512u + (i & 511u)) * 8u) =
                        make_uint2(__builtin_bit_cast(uint32_t, a * f), __builtin_bit_cast(uint32_t, b * f));
                }
            } else {
                const H8 base = entry_halves<fmt<SRC>() != F_XXS>(e[n]);
#pragma unroll
                for (uint32_t k = 0; k < (fmt<SRC>() == F_M ? 2u : 4u); ++k) {
                    const uint32_t at = fmt<SRC>() == F_M ? 2048u * k + i : 4u * i + ((k + (i >> 2)) & 3u);
                    H8 v = base;
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        if constexpr (fmt<SRC>() == F_XXS) { const half2_t f = odd_halves(at & 15u); v.p[p] = base.p[p] * f; }
                        if constexpr (fmt<SRC>() == F_M) { const _Float16 off = k ? -0.125f : 0.125f; v.p[p] = base.p[p] + half2_t{off, off}; }      // (exact: a byte and three bits behind the point)
                    }
                    *reinterpret_cast<uint4 *>(entries + at * 16u) = v.u;
                }
            }
        }
    }
};

// The small tables, by T threads in two parts: a thread's codebook entries are requested (before the rows, which the second part must not
// wait for), then written. Tables with copies are written by two threads per entry, half of the copies each.
template <int SRC> constexpr uint32_t small_copies() { return fmt<SRC>() == F_XXS ? 8u : fmt<SRC>() == F_M ? 1u : 4u; }
template <int SRC> constexpr uint32_t entry_shift() { return !small_tables<SRC>() ? (fmt<SRC>() == F_M ? 4u : 7u) : fmt<SRC>() == F_XXS ? 7u : fmt<SRC>() == F_XS ? 6u : fmt<SRC>() == F_M ? 4u : 5u; }
template <int SRC> constexpr uint32_t small_entry_bytes() { return codebook_entries<SRC>() << entry_shift<SRC>(); }
template <int SRC, uint32_t T> struct SmallSeeds {
    static constexpr uint32_t kHalves = small_copies<SRC>() > 1u ? 2u : 1u, kItems = codebook_entries<SRC>() * kHalves, N = (kItems + T - 1u) / T;
    uint64_t e[N];
    __device__ __forceinline__ void request(uint32_t tid, const int8_t *grid) {
#pragma unroll
        for (uint32_t n = 0; n < N; ++n) {
            const uint32_t i = (min(tid + n * T, kItems - 1u)) / kHalves;
            if constexpr (is_iq3<SRC>()) e[n] = redhip_iq3s_grid[i];
            else if constexpr (fmt<SRC>() == F_XXS) e[n] = redhip_iq2xxs_grid[i];
            else e[n] = reinterpret_cast<const uint64_t *>(grid)[i];
        }
    }
    __device__ __forceinline__ void store(uint8_t *entries, uint32_t *signs, uint32_t tid) const {
        constexpr uint32_t kCopies = small_copies<SRC>(), kMine = kCopies / kHalves;
#pragma unroll
        for (uint32_t n = 0; n < N; ++n) {
            const uint32_t i = min(tid + n * T, kItems - 1u), first = ((i / kHalves) * kCopies + (i % kHalves) * kMine);      // (surplus threads repeat the last)
            if constexpr (is_iq3<SRC>()) {
                const uint2 v = make_uint2(__builtin_bit_cast(uint32_t, byte_halves<0u, false>((uint32_t)e[n])), __builtin_bit_cast(uint32_t, byte_halves<2u, false>((uint32_t)e[n])));
#pragma unroll
                for (uint32_t c = 0; c < kMine; ++c) *reinterpret_cast<uint2 *>(entries + (size_t)(first + c) * 8u) = v;
            } else {
                const H8 v = entry_halves<fmt<SRC>() != F_XXS>(e[n]);
#pragma unroll
                for (uint32_t c = 0; c < kMine; ++c) *reinterpret_cast<uint4 *>(entries + (size_t)(first + c) * 16u) = v.u;
            }
        }
        build_signs<SRC, T>(signs, tid);
    }
};

// fields of a quarter block (two 32-column groups) of a row: what a lane multiplies
//   IQ2_XXS  a: the two groups' words                     IQ2_XS  a: eight 16-bit entries, c: two scale bytes
//   IQ1_M    a: 8 index bytes | 4 bytes of nibbles | scale word     IQ3_S   a: 16 index bytes, b: 8 sign bytes, c: two qh bytes | scale byte << 16
//   tile-major IQ3_S   a, b: entry q of the first and the last four groups of the block, a word each
struct Quarter { uint4 a, b; uint32_t c; };

template <class T> __device__ __forceinline__ T load_a2(const uint8_t *p) { T v; __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), sizeof(T)); return v; }

// Quarter q of block kc of row r of a tile of 16 rows, and what its d is made from. tile: the tile's rows (raw and packed rows 16 KP blocks,
// tile-major its KP * 2 chunks of 16 rows), ds: its block scales, scs: tile-major IQ2_XS, its scale bytes.
//   tile-major: chunk c (128 columns) of row r at (c * 16 + r) * 32 (IQ3_S words * 64), scale of block b at (b * 16 + r) * 2, the scale
//   bytes of a chunk at (c * 16 + r) * 4: a wave's load is two runs of 512 bytes
template <int SRC, uint32_t KP>
__device__ __forceinline__ void load_quarter(const uint8_t *tile, const uint8_t *ds, const uint8_t *scs, uint32_t r, uint32_t kc, uint32_t q, Quarter &v, uint2 &d) {
    const uint32_t block = r * KP + kc;
    if constexpr (layout<SRC>() == L_TILED) {
        const uint32_t chunk = (2u * kc + (q >> 1)) * 16u + r;
        if constexpr (fmt<SRC>() == F_IQ3_WORDS) {
            v.a = *reinterpret_cast<const uint4 *>(tile + (32u * kc + r) * 64u + 16u * q);
            v.b = *reinterpret_cast<const uint4 *>(tile + (32u * kc + 16u + r) * 64u + 16u * q);
        } else if constexpr (fmt<SRC>() == F_M) {      // stream words: four index bytes | nibbles, two 3-bit scales from bit 16 on
            const uint4 w = *reinterpret_cast<const uint4 *>(tile + chunk * 32u + 16u * (q & 1u));
            v.a = make_uint4(w.x, w.z, (w.y & 0xffffu) | (w.w << 16), __builtin_amdgcn_ubfe(w.y, 16u, 6u) | (__builtin_amdgcn_ubfe(w.w, 16u, 6u) << 6));
        } else
            v.a = *reinterpret_cast<const uint4 *>(tile + chunk * 32u + 16u * (q & 1u));
        if constexpr (fmt<SRC>() == F_XS) v.c = *reinterpret_cast<const uint16_t *>(scs + each_trip(chunk * 32u + 16u * (q & 1u)) / 8u);      // (no register of its own beside the quarter's)
        d.x = *reinterpret_cast<const uint16_t *>(ds + (kc * 16u + r) * 2u);
    } else if constexpr (layout<SRC>() == L_ROWS) {
        v.a = *reinterpret_cast<const uint4 *>(tile + block * 64u + 16u * q);
        d.x = *reinterpret_cast<const uint16_t *>(ds + block * 2u);
    } else {
        const uint8_t *bp = tile + block * src_block<SRC>();
        if constexpr (fmt<SRC>() == F_M && layout<SRC>() == L_RAW) {
            const uint2 qs = load_a2<uint2>(bp + 8u * q);
            v.a = make_uint4(qs.x, qs.y, load_a2<uint32_t>(bp + 32u + 4u * q), load_a2<uint16_t>(bp + 48u + 2u * q));
            d = load_a2<uint2>(bp + 48u);
        } else {
            v.a = load_a2<uint4>(bp + 2u + 16u * q);
            d.x = load_a2<uint16_t>(bp);
        }
        if constexpr (fmt<SRC>() == F_XS) v.c = load_a2<uint16_t>(bp + 66u + 2u * q);
        if constexpr (fmt<SRC>() == F_IQ3) {
            const uint2 sg = load_a2<uint2>(bp + 74u + 8u * q);
            v.b.x = sg.x; v.b.y = sg.y;
            v.c = load_a2<uint16_t>(bp + 66u + 2u * q) | ((uint32_t)bp[106u + q] << 16);
        }
    }
}
template <int SRC>
__device__ __forceinline__ float quarter_d(uint2 d) {
    if constexpr (fmt<SRC>() == F_M && layout<SRC>() == L_RAW) return scale_to_f32(((d.x >> 12) & 0x000fu) | ((d.x >> 24) & 0x00f0u) | ((d.y >> 4) & 0x0f00u) | ((d.y >> 16) & 0xf000u));
    else return scale_to_f32(d.x);
}

// odd integer 2 s + 1 as two equal fp16 halves, s the BITS bits of w at AT: 1024 + (2 s + 1) by integer arithmetic, minus 1024, exact
template <uint32_t AT, uint32_t BITS> __device__ __forceinline__ half2_t odd_splat(uint32_t w) {
    const uint32_t big = and_or(moved<AT, 1u>(w), (2u << BITS) - 2u, 0x6401u);
    const _Float16 h = __builtin_bit_cast(_Float16, (uint16_t)big);
    return half2_t{h, h} - half2_t{(_Float16)1024.0f, (_Float16)1024.0f};
}

// f(constant 0) .. f(constant 7): the steps of a quarter block
template <class F, uint32_t... S> __device__ __forceinline__ void each_step_of(F &&f, std::integer_sequence<uint32_t, S...>) { (f(std::integral_constant<uint32_t, S>{}), ...); }
template <uint32_t N, class F> __device__ __forceinline__ void each(F &&f) { each_step_of(f, std::make_integer_sequence<uint32_t, N>{}); }
template <class F> __device__ __forceinline__ void each_step(F &&f) { each_step_of(f, std::make_integer_sequence<uint32_t, 8>{}); }

// lane constants of the tables: addresses of the lane's copy, masks in vector registers
struct LaneTables {
    const uint8_t *entries, *signs;        // (signs: the lane's copy is or-ed into the offset)
    uint32_t entry_mask, sign_mask, sign_lane, scale_mask, sign_bits;
};
template <int SRC> constexpr uint32_t entry_copies() { return small_tables<SRC>() ? small_copies<SRC>() : fmt<SRC>() == F_XS ? 8u : 1u; }
template <int SRC> __device__ __forceinline__ LaneTables lane_tables(const uint8_t *entries, const uint32_t *signs, uint32_t tid) {
    constexpr uint32_t C = sign_copies<SRC>() ? sign_copies<SRC>() : 1u, E = is_iq3<SRC>() ? 8u : 16u, ES = entry_shift<SRC>();
    LaneTables t;
    t.entries = entries + (tid % entry_copies<SRC>()) * E;
    t.signs = reinterpret_cast<const uint8_t *>(signs);
    t.sign_lane = (tid % C) * 4u;
    t.sign_mask = in_vector((is_iq3<SRC>() ? 255u : 127u) << sign_shift<SRC>());
    t.entry_mask = in_vector(fmt<SRC>() == F_XS ? 511u << ES : fmt<SRC>() == F_XXS ? 255u << ES : fmt<SRC>() == F_M ? 255u << ES : fmt<SRC>() == F_IQ3_WORDS ? 0xff8u : 255u << 3);
    t.scale_mask = in_vector(0xf000u);
    t.sign_bits = in_vector(0x80008000u);
    return t;
}

// Table reads of step s (eight columns) of a quarter, then the arithmetic on what they return: the eight signed, scaled fp16 weights.
struct Entry { uint4 m; uint32_t s; };
__device__ __forceinline__ uint32_t word_of(const uint4 &v, uint32_t i) { return i == 0u ? v.x : i == 1u ? v.y : i == 2u ? v.z : v.w; }
template <int SRC, uint32_t S>
__device__ __forceinline__ Entry fetch_entry(const Quarter &v, const LaneTables &t) {
    constexpr uint32_t h = S >> 2, e = S & 3u, ES = entry_shift<SRC>(), SS = sign_shift<SRC>();                 // group of the quarter, entry of the group
    const auto entry = [&](uint32_t off) { return *reinterpret_cast<const uint4 *>(t.entries + off); };
    const auto half_entry = [&](uint32_t off) { return *reinterpret_cast<const uint2 *>(t.entries + off); };
    const auto sign = [&](uint32_t w) { return *reinterpret_cast<const uint32_t *>(t.signs + and_or(w, t.sign_mask, t.sign_lane)); };
    Entry r;
    if constexpr (fmt<SRC>() == F_XXS) {
        const uint32_t wa = h ? v.a.z : v.a.x, wb = h ? v.a.w : v.a.y;
        // bytes 0 .. 3 of the permute's second operand are the entries, 7 the top byte of the first
        if constexpr (small_tables<SRC>()) r.m = entry(moved<8u * e, ES>(wa) & t.entry_mask);
        else r.m = entry(__builtin_amdgcn_perm(wb & 0xf0000000u, wa, 0x0c0c0007u | (e << 8)));
        r.s = sign(moved<7u * e, SS>(wb));
    } else if constexpr (fmt<SRC>() == F_XS) {
        const uint32_t w = word_of(v.a, 2u * h + (e >> 1));
        constexpr uint32_t o = 16u * (e & 1u);
        r.m = entry(moved<o, ES>(w) & t.entry_mask);
        r.s = sign(moved<o + 9u, SS>(w));
    } else if constexpr (fmt<SRC>() == F_IQ3_WORDS) {
        const uint32_t w = word_of(h ? v.b : v.a, e), top = w >> 14, scale = top & t.scale_mask;      // nibble * 512 entries * 8 bytes
        const uint2 ma = half_entry(and_or(w << 3, t.entry_mask, scale)), mb = half_entry(and_or(w >> 6, t.entry_mask, scale));
        r.m = make_uint4(ma.x, ma.y, mb.x, mb.y);
        r.s = sign(top);
    } else if constexpr (fmt<SRC>() == F_M) {
        const uint32_t idx = h ? v.a.y : v.a.x;
        if constexpr (small_tables<SRC>()) {
            r.s = __builtin_amdgcn_ubfe(v.a.z, 16u * h + 4u * e, 4u);
            r.m = entry((__builtin_amdgcn_ubfe(idx, 8u * e, 8u) | ((r.s & 7u) << 8)) << ES);
        } else {
            r.s = 0u;
            r.m = entry(and_or(moved<8u * e, 4u>(idx), t.entry_mask, moved<16u * h + 4u * e, 12u>(v.a.z) & t.scale_mask));
        }
    } else {
        const uint32_t w = word_of(v.a, 2u * h + (e >> 1));
        constexpr uint32_t o = 16u * (e & 1u), ba = 8u * h + 2u * e, bb = ba + 1u;     // qh bits of the two entries -> bit 11
        const uint32_t scale = moved<h ? 20u : 16u, 12u>(v.c) & t.scale_mask;      // nibble * 512 entries * 8 bytes
        const uint32_t ha = moved<ba, 11u>(v.c) & 2048u, hb = moved<bb, 11u>(v.c) & 2048u;
        uint32_t ia = and_or(moved<o, 3u>(w), t.entry_mask, ha), ib = and_or(moved<o + 8u, 3u>(w), t.entry_mask, hb);      // entry * 8
        if constexpr (small_tables<SRC>()) { ia <<= 2; ib <<= 2; }
        else { ia |= scale; ib |= scale; }
        const uint2 ma = half_entry(ia), mb = half_entry(ib);
        r.m = make_uint4(ma.x, ma.y, mb.x, mb.y);
        r.s = sign(moved<8u * e, SS>(h ? v.b.y : v.b.x));
    }
    return r;
}
// f: the scale of the step's columns where the table does not hold it (sixteen columns IQ2_XS, IQ1_M; 32 the others, small tables)
template <int SRC> constexpr uint32_t steps_per_scale() { return fmt<SRC>() == F_XS || fmt<SRC>() == F_M ? 2u : small_tables<SRC>() ? 4u : 0u; }
template <int SRC, uint32_t S>
__device__ __forceinline__ half2_t step_scale(const Quarter &v) {
    constexpr uint32_t h = S >> 2, e = S & 3u;
    if constexpr (fmt<SRC>() == F_XS) return odd_splat<8u * h + 4u * (e >> 1), 4u>(v.c);
    else if constexpr (fmt<SRC>() == F_M) return odd_splat<6u * h + 3u * (e >> 1), 3u>(v.a.w);
    else if constexpr (fmt<SRC>() == F_XXS) return odd_splat<28u, 4u>(h ? v.a.w : v.a.y);
    else return odd_splat<16u + 4u * h, 4u>(v.c);
}
template <int SRC>
__device__ __forceinline__ half8_t finish_entry(const Entry &e, half2_t f, const LaneTables &t) {
    H8 r;
    r.u = e.m;
    if constexpr (fmt<SRC>() == F_M && !small_tables<SRC>()) {
#pragma unroll
        for (int i = 0; i < 4; ++i) r.p[i] = r.p[i] * f;
    } else if constexpr (fmt<SRC>() == F_M) {
        // (2 s + 1) / 8 with the sign of the offset: three exponent steps down (2 s + 1 >= 1 is a normal number), sign bit by xor
        const uint32_t neg = (e.s & 8u) << 12;
        const half2_t off = __builtin_bit_cast(half2_t, (__builtin_bit_cast(uint32_t, f) - 0x0c000c00u) ^ (neg | (neg << 16)));
#pragma unroll
        for (int i = 0; i < 4; ++i) r.p[i] = r.p[i] * f + off;
    } else {
        // (the one-token kernels, which have the small tables, wait for this chain: two doublings at most in a row, the second step a shift)
        const uint32_t s1 = twice(e.s), s2 = small_tables<SRC>() ? e.s << 2 : twice(s1), s3 = twice(s2);
        if constexpr (fmt<SRC>() == F_XS || small_tables<SRC>()) {     // IQ2_XS entries are signed bytes in general: the sign goes to the (positive) scale
            const uint32_t fb = __builtin_bit_cast(uint32_t, f);
            r.p[0] *= __builtin_bit_cast(half2_t, and_or(e.s, t.sign_bits, fb));
            r.p[1] *= __builtin_bit_cast(half2_t, and_or(s1, t.sign_bits, fb));
            r.p[2] *= __builtin_bit_cast(half2_t, and_or(s2, t.sign_bits, fb));
            r.p[3] *= __builtin_bit_cast(half2_t, and_or(s3, t.sign_bits, fb));
        } else
            r.u = make_uint4(and_or(e.s, t.sign_bits, e.m.x), and_or(s1, t.sign_bits, e.m.y), and_or(s2, t.sign_bits, e.m.z), and_or(s3, t.sign_bits, e.m.w));
    }
    return r.v;
}

}  // namespace redhip
