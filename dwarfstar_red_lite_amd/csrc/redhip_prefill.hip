// What a chunk of tokens (prefill) needs beside its tile kernels (redhip_tiles.hip): the tile lists, the tile-major copies of the experts'
// matrices, and dense f32 products on the bf16 matrix units, three terms for each f32 (router logits, the shared expert of mixed layouts).
#include <hip/hip_runtime.h>

#include "redhip_mfma.h"

#include <type_traits>

namespace redhip {

// ---------------------------------------------------------------- tile list

// the tile lists (TileLists) as a launch of their own, for callers whose pair sort did not write them
__global__ __launch_bounds__(1024) void build_tiles_kernel(const uint32_t *uid, const uint32_t *expert_start, const uint32_t *n_unique, uint32_t P, TileLists tl) {
    __shared__ uint32_t wave_total[3][16];
    const uint32_t tid = threadIdx.x, U = n_unique[0];
    uint32_t e = 0u, p0 = 0u, n = 0u;
    if (tid < U) { e = uid[tid]; p0 = expert_start[tid]; n = expert_start[tid + 1u] - p0; }
    build_tile_lists(e, p0, n, P, tl, wave_total);
}

hipError_t launch_build_tiles(const uint32_t *uid, const uint32_t *expert_start, const uint32_t *n_unique, uint32_t n_pairs, const TileLists &tl, hipStream_t s) {
    REDHIP_LAUNCH(build_tiles_kernel, dim3(1), dim3(1024), 0, s, uid, expert_start, n_unique, n_pairs, tl);
    return hipGetLastError();
}

// ---------------------------------------------------------------- tile-major copies

// The 32-byte chunks (four groups of 32 columns) of 16 consecutive rows of a packed matrix lie next to each other, so that one wave-wide
// load of the tile kernels is two runs of 512 contiguous bytes:
//   chunk (row, c)  at ((row / 16 * (K / 128) + c) * 16 + row % 16) * 32          c = chunk of four groups along K
//   scale (row, b)  at qs_bytes + ((row / 16 * (K / 256) + b) * 16 + row % 16) * 2
// row-major packed matrix -> tile-major copy; one thread per 32-byte chunk, the scales ride along (with_sc: an IQ2_XS stream, whose scale
// bytes [row][group] follow qs and ds; the four of a chunk become one 32-bit word at (tile, chunk, row) like the chunk itself)
__global__ void tile_packed_kernel(const uint8_t *packed, uint64_t packed_stride, uint32_t nrows, uint32_t K, uint8_t *tiled, uint64_t tiled_stride, int with_sc) {
    const uint32_t NC = K / 128u, NB = K / 256u;
    const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (uint64_t)nrows * NC) return;
    const uint32_t row = (uint32_t)(gid / NC), c = (uint32_t)(gid % NC);
    const uint8_t *src = packed + (uint64_t)blockIdx.y * packed_stride;
    uint8_t *dst = tiled + (uint64_t)blockIdx.y * tiled_stride;
    const uint64_t qs_bytes = (uint64_t)nrows * (K / 32u) * 8u;
    const uint4 *sp = reinterpret_cast<const uint4 *>(src + ((uint64_t)row * (K / 32u) + 4u * c) * 8u);
    uint4 *dp = reinterpret_cast<uint4 *>(dst + (((uint64_t)(row / 16u) * NC + c) * 16u + row % 16u) * 32u);
    dp[0] = sp[0];
    dp[1] = sp[1];
    if ((c & 1u) == 0u) {
        const uint32_t b = c / 2u;
        reinterpret_cast<uint16_t *>(dst + qs_bytes)[((uint64_t)(row / 16u) * NB + b) * 16u + row % 16u] =
            reinterpret_cast<const uint16_t *>(src + qs_bytes)[(uint64_t)row * NB + b];
    }
    if (with_sc) {
        const uint64_t sc_off = qs_bytes + (uint64_t)nrows * NB * 2u;
        reinterpret_cast<uint32_t *>(dst + sc_off)[((uint64_t)(row / 16u) * NC + c) * 16u + row % 16u] =
            *reinterpret_cast<const uint32_t *>(src + sc_off + (uint64_t)row * (K / 32u) + 4u * c);
    }
}

hipError_t launch_tile_packed(const void *packed, uint64_t packed_stride, uint32_t count, uint32_t nrows, uint32_t K, void *tiled, uint64_t tiled_stride,
                              hipStream_t s, bool with_sc) {
    if (!nrows || nrows % 16u || !K || K % 256u || !count || count > 65535u) return hipErrorInvalidValue;
    const uint64_t total = (uint64_t)nrows * (K / 128u);
    REDHIP_LAUNCH(tile_packed_kernel, dim3((uint32_t)((total + 255u) / 256u), count), dim3(256), 0, s, static_cast<const uint8_t *>(packed), packed_stride,
                  nrows, K, static_cast<uint8_t *>(tiled), tiled_stride, with_sc ? 1 : 0);
    return hipGetLastError();
}

// Tile-major IQ3_S (built once at upload from the raw 110-byte blocks): per group of 32 weights four 32-bit words, one per eight
// weights l: bits 0-8 the first grid index, 9-17 the second (each with its ninth bit from qh), 18-25 the eight sign bits, 26-29 the
// group's scale nibble. A row's chunk of four groups is stored as [l][group] so that lane (r, l) reads its own four words as one
// 16-byte load, and the chunks of 16 consecutive rows lie next to each other (a wave-wide load is 1024 contiguous bytes):
//   chunk (row, c)  at ((row / 16 * (K / 128) + c) * 16 + row % 16) * 64,   lane l adds 16 l
//   scale (row, b)  at qs_bytes + ((row / 16 * (K / 256) + b) * 16 + row % 16) * 2
__global__ void tile_iq3s_kernel(const uint8_t *raw, uint64_t raw_stride, uint32_t nrows, uint32_t K, uint8_t *tiled, uint64_t tiled_stride) {
    const uint32_t NG = K / 32u, NC = K / 128u, NB = K / 256u;
    const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (uint64_t)nrows * NG) return;
    const uint32_t row = (uint32_t)(gid / NG), g = (uint32_t)(gid % NG), sub = g & 7u;
    const uint8_t *bp = raw + (uint64_t)blockIdx.y * raw_stride + ((uint64_t)row * NB + (g >> 3)) * 110u;
    uint8_t *dst = tiled + (uint64_t)blockIdx.y * tiled_stride;
    const uint32_t nib = ((uint32_t)bp[106u + (sub >> 1)] >> (4u * (sub & 1u))) & 15u, qh = bp[66u + sub];
    uint32_t *out = reinterpret_cast<uint32_t *>(dst + (((uint64_t)(row / 16u) * NC + (g >> 2)) * 16u + row % 16u) * 64u);
    for (uint32_t l = 0; l < 4u; ++l) {
        const uint32_t ia = (uint32_t)bp[2u + 8u * sub + 2u * l] | ((qh << (8u - 2u * l)) & 256u);
        const uint32_t ib = (uint32_t)bp[3u + 8u * sub + 2u * l] | ((qh << (7u - 2u * l)) & 256u);
        out[4u * l + (g & 3u)] = ia | (ib << 9) | ((uint32_t)bp[74u + 4u * sub + l] << 18) | (nib << 26);
    }
    if (sub == 0u)
        reinterpret_cast<uint16_t *>(dst + (uint64_t)nrows * NG * 16u)[((uint64_t)(row / 16u) * NB + (g >> 3)) * 16u + row % 16u] = (uint16_t)ld_u16(bp);
}

hipError_t launch_tile_iq3s(const void *raw, uint64_t raw_stride, uint32_t count, uint32_t nrows, uint32_t K, void *tiled, uint64_t tiled_stride, hipStream_t s) {
    if (!nrows || nrows % 16u || !K || K % 256u || !count || count > 65535u) return hipErrorInvalidValue;
    const uint64_t total = (uint64_t)nrows * (K / 32u);
    REDHIP_LAUNCH(tile_iq3s_kernel, dim3((uint32_t)((total + 255u) / 256u), count), dim3(256), 0, s, static_cast<const uint8_t *>(raw), raw_stride, nrows, K,
                  static_cast<uint8_t *>(tiled), tiled_stride);
    return hipGetLastError();
}

// ---------------------------------------------------------------- router logits of a token chunk

// out[tok][row] = W[row] . x[tok] for an f32 matrix W (a router, the dense shared expert of mixed layouts) and a chunk of activations. Every f32
// is the sum of three bf16 numbers, exactly (the nearest one, the nearest to the rest, and what is left), and of the
// nine products of such sums (a published way to f32 products: Henry, Tang, Heinecke, ARITH 2019) the six that reach 2^-24 of the largest go through v_mfma_f32_16x16x32_bf16: six of those are 96 cycles for 32 columns
// where the fp32 unit takes 256. The products of the leading terms have accumulators of their own, the other five share one.
// A workgroup owns BR = 16 MR rows x BT = 16 MT tokens, each of its eight waves an eighth of k for all of them; the eight sums meet in LDS, in
// double. A wave fetches 32 columns of every row and token straight into LDS (full 128-byte lines: sixteen lanes of a load that name sixteen rows
// take four times as long, 26 instead of 15 us for 64 x 32 outputs of 2048 columns), takes them into registers as fragments (lane (r = l % 16, q = l / 16):
// columns 4q .. 4q + 3 and 16 + 4q .. of row r; the 16-byte pieces of a row are permuted by r / 2 so that a read pass meets every bank once),
// requests the next 32 columns into the same place and multiplies meanwhile. No barrier before the sums meet.
// What bounds it: the fetch - 96 KB in flight for a tile of 64 x 32, which cover about the 1 .. 1.5 us that they take - then splitting and multiplying
// (2300 .. 3000 cycles for each 256 columns). us, before (v_mfma_f32_16x16x4_f32, both operands through registers into LDS) -> now:
// gate/up with SwiGLU of 1024 x 2048: 77 tokens 12.3 -> 8.2, 512: 31 -> 20, 2048: 94 -> 83; down 2048 x 512: 77 tokens 6.7 -> 5.0, 512: 16.6 -> 15,
// 2048: 57 -> 57; router 512 x 2048: 77 tokens 10.4 -> 8.2, 512: 18.7 -> 12.7, 2048: 47 -> 41.
// The order in which an output's products are added is the same for every tile. Error against a sum in double, of the rms of the outputs: 2048
// columns 0.74e-7 (two chains of leading products a wave), 512 columns 0.53e-7, where the fp32 unit with totals in double left 1.04e-7 and 1.1e-7 (and
// 4.1e-7 in a router's plain chains); gate and up products multiplied by SwiGLU 1.1 .. 1.3e-7, 1.6e-7 before. Terms that are cut instead of rounded are
// a fifth cheaper to make, but leave out products that all have the sign of the whole: 0.94e-7, and twice that where one product outweighs the rest.
// An infinity or NaN has no three terms, and an infinite sum may come out as NaN: a tile with outputs that are not finite multiplies once more, on the
// fp32 unit, for these. (An output at a time, a thread's 2048 products behind one another, a chunk of 512 tokens of NaN took 3.2 ms an F2 layer; now 0.30,
// of numbers 0.28. Where only a leading term overflows 3e-7 .. 4e-7 are lost, 6.6e-7 then.)
// SWIGLU: W holds gate rows, then as many up rows; the upper half of a tile's row blocks are gate rows, the lower half the up rows of the same
// columns, and out gets silu(gate) * up of them: no pass of its own over the products.
// Launches with xh get workgroups behind the tiles that write the fp16 halves of the activations (a wave per token, split_token) and multiply them
// with gate_inp, if there is one, as row n_rows; without xh the tiles have it as a further row.

__device__ __forceinline__ void split_token(const float *gate_inp, const float *x, float *logits, uint32_t out_stride, _Float16 *xh, _Float16 *xl, int *xexp, uint32_t H,
                                            uint32_t E, uint32_t tok, uint32_t lane, float *scalar = nullptr) {
            // the vector as float4 per lane, eight requested at a time (2048 elements per pass: one round trip for the usual widths)
            const float4 *xt = reinterpret_cast<const float4 *>(x + (uint64_t)tok * H), *gv = reinterpret_cast<const float4 *>(gate_inp);
            const uint32_t H4 = H / 4u;
            float amax = 0.0f, gate = 0.0f;
            for (uint32_t base = 0; base < H4; base += 512u) {
                float4 v[8], g[8];
    #pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint32_t i = base + 64u * k + lane;
                    v[k] = i < H4 ? xt[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    g[k] = gate_inp && i < H4 ? gv[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                }
    #pragma unroll
                for (int k = 0; k < 8; ++k) {
                    amax = fmaxf(fmaxf(amax, fmaxf(fabsf(v[k].x), fabsf(v[k].y))), fmaxf(fabsf(v[k].z), fabsf(v[k].w)));
                    gate = fmaf(g[k].w, v[k].w, fmaf(g[k].z, v[k].z, fmaf(g[k].y, v[k].y, fmaf(g[k].x, v[k].x, gate))));
                }
            }
    #pragma unroll
            for (int o = 32; o > 0; o >>= 1) { amax = fmaxf(amax, __shfl_xor(amax, o, 64)); gate += __shfl_xor(gate, o, 64); }
            const int e = prescale_exp(amax);
            const float inv = exp2i(-e);
            for (uint32_t base = 0; base < H4; base += 512u) {
                float4 v[8];
    #pragma unroll
                for (int k = 0; k < 8; ++k) { const uint32_t i = base + 64u * k + lane; v[k] = xt[i < H4 ? i : 0u]; }
    #pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint32_t i = base + 64u * k + lane;
                    if (i >= H4) continue;
                    const float f[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
                    half4_t h4, l4;
    #pragma unroll
                    for (int c = 0; c < 4; ++c) { _Float16 hh, ll; split_hi_lo(f[c], inv, &hh, &ll); h4[c] = hh; l4[c] = ll; }
                    *reinterpret_cast<half4_t *>(xh + (uint64_t)tok * H + 4u * i) = h4;
                    *reinterpret_cast<half4_t *>(xl + (uint64_t)tok * H + 4u * i) = l4;
                }
            }
            if (lane == 0u) {
                xexp[tok] = e;
                if (scalar) scalar[tok] = 1.0f / (1.0f + expf(-gate));
                else if (gate_inp) logits[(uint64_t)tok * out_stride + E] = gate;
            }
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint32x4_t __attribute__((ext_vector_type(4)));
struct ThreeTerms { bf16x8 high, mid, low; };
// `top` = 0xffff0000, `half` = 0x8000 in vector registers
__device__ __forceinline__ ThreeTerms three_terms(float4_t a, float4_t b, uint32_t top, uint32_t half) {
    const auto near = [&](float v) { return __uint_as_float((__float_as_uint(v) + half) & top); };      // (a NaN may lose its mark here; the last term keeps it)
    const auto tops = [](float v1, float v0) { return __builtin_amdgcn_perm(__float_as_uint(v1), __float_as_uint(v0), 0x07060302u); };
    uint32x4_t h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v0 = i < 2 ? a[2 * (i & 1)] : b[2 * (i & 1)], v1 = i < 2 ? a[2 * (i & 1) + 1] : b[2 * (i & 1) + 1];
        const float h0 = near(v0), h1 = near(v1), r0 = v0 - h0, r1 = v1 - h1, m0 = near(r0), m1 = near(r1);      // (each difference exact)
        h[i] = tops(h1, h0);
        m[i] = tops(m1, m0);
        l[i] = tops(r1 - m1, r0 - m0);
    }
    return ThreeTerms{__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

// what a kernel of both kinds multiplies beside its gate and up rows: a router (n_rows may be 0); `scalar`: the shared expert's gate factor instead of row n_rows
struct RouterRows { const float *w; float *out, *scalar; uint32_t n_rows, out_stride; };
enum F32Kind { F32_PLAIN, F32_SWIGLU, F32_BOTH };
template <F32Kind KIND> struct Beside {};
template <> struct Beside<F32_BOTH> : RouterRows {};

template <int MR, int MT, F32Kind KIND>
__global__ __launch_bounds__(512) void f32_tiles_kernel(const float *w, const float *gate_inp, const float *x, float *out, uint32_t out_stride, _Float16 *xh,
                                                        _Float16 *xl, int *xexp, uint32_t K, uint32_t n_rows, uint32_t ntok, Beside<KIND> router) {
    constexpr uint32_t BR = 16u * MR, BT = 16u * MT, NB = MR + MT, PIECES = 2u * NB > MR * MT ? 2u * NB : MR * MT;      // KB per wave: 32 columns of the rows and tokens, later its sums
    __shared__ __attribute__((aligned(16))) float4_t lds[8][PIECES][64];
    __shared__ uint32_t again;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t tok_tiles = (ntok + BT - 1u) / BT, first = KIND == F32_BOTH ? n_rows / BR * tok_tiles : 0u;      // tiles of gate and up rows in front of the router's
    const bool swiglu = KIND == F32_SWIGLU || (KIND == F32_BOTH && blockIdx.x < first);
    uint32_t tile = blockIdx.x;
    if constexpr (KIND == F32_BOTH)
        if (!swiglu) { tile -= first; w = router.w; n_rows = router.n_rows; out = router.out; out_stride = router.out_stride; }
    const uint32_t all_rows = n_rows + (gate_inp && !xh ? 1u : 0u), row_tiles = (all_rows + BR - 1u) / BR;
    if (tile >= row_tiles * tok_tiles) {
        const uint32_t tok = 8u * (tile - row_tiles * tok_tiles) + wave;
        float *scalar = nullptr;
        if constexpr (KIND == F32_BOTH) scalar = router.scalar;
        if (tok < ntok) split_token(gate_inp, x, out, out_stride, xh, xl, xexp, K, n_rows, tok, lane, scalar);
        return;
    }
    // Workgroups are dealt to the eight XCDs in turn, each with its own L2: workgroup i lands on XCD i % 8. The tiles of one XCD form a
    // compact block of the tile grid (a quarter of the row tiles x half of the token tiles), so that an XCD fetches a quarter of the
    // matrix and half of the activations instead of all of both. (A different dealing order would only cost this locality.)
    uint32_t tile_r = tile % row_tiles, tile_t = tile / row_tiles;
    if (row_tiles % 4u == 0u && tok_tiles % 2u == 0u) {
        const uint32_t xcd = tile & 7u, slot = tile >> 3, br = row_tiles / 4u, bt = tok_tiles / 2u;
        tile_r = (xcd & 3u) * br + slot % br;
        tile_t = (xcd >> 2) * bt + slot / br;
    }
    // row block m of the tile starts here; rows and tokens beyond the last repeat another and are not stored
    const auto block_row = [&](uint32_t m) { return swiglu ? (m < MR / 2u ? 0u : n_rows / 2u) + tile_r * (BR / 2u) + 16u * (m % (MR / 2u)) : tile_r * BR + 16u * m; };
    const auto matrix_row = [&](uint32_t row) { return row < n_rows ? w + (uint64_t)row * K : gate_inp ? gate_inp : w; };
    // fetch i of a wave: eight rows (or tokens) of 128 bytes; lane l brings piece (l % 8) ^ (row % 16 / 2) of row l / 8
    const float *src[2u * NB];
#pragma unroll
    for (uint32_t i = 0; i < 2u * NB; ++i) {
        const uint32_t l = 8u * (i & 1u) + (lane >> 3);
        src[i] = i < 2u * MR ? matrix_row(block_row(i / 2u) + l) : x + (uint64_t)min(tile_t * BT + 16u * (i / 2u - MR) + l, ntok - 1u) * K;
        src[i] += K / 8u * wave + 4u * ((lane & 7u) ^ (l >> 1));
    }
    float4_t *mine = &lds[wave][0][0];
    const bool in_pieces = (reinterpret_cast<uintptr_t>(x) & 15u) == 0u;      // (the caller's activations may lie at any float)
    const auto request = [&](uint32_t step) {
        if (in_pieces) {
#pragma unroll
            for (uint32_t i = 0; i < 2u * NB; ++i)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src[i] + 32u * step), (__attribute__((address_space(3))) void *)(mine + 64u * i), 16, 0, 0);
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 2u * NB; ++i) {
                const float *p = src[i] + 32u * step;
                mine[64u * i + lane] = float4_t{p[0], p[1], p[2], p[3]};
            }
        }
    };
    float4_t high[2][MR][MT], low[MR][MT];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int t = 0; t < MT; ++t) high[0][m][t] = high[1][m][t] = low[m][t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t top = in_vector(0xffff0000u), half = in_vector(0x8000u), at0 = 8u * r + (q ^ (r >> 1)), at1 = 8u * r + ((q + 4u) ^ (r >> 1)), steps = K / 256u;
    const auto fetched = [&](uint32_t step, float4_t (&v)[NB][2]) {      // this step's columns into registers, the next ones requested
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // they are in LDS
#pragma unroll
        for (uint32_t i = 0; i < NB; ++i) { v[i][0] = mine[128u * i + at0]; v[i][1] = mine[128u * i + at1]; }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // and read, before the next ones take their place
        if (step + 1u < steps) request(step + 1u);
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto multiply = [&](uint32_t step, auto chain) {
        constexpr int C = decltype(chain)::value;
        float4_t v[NB][2];
        fetched(step, v);
        ThreeTerms b[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) b[t] = three_terms(v[MR + t][0], v[MR + t][1], top, half);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            const ThreeTerms a = three_terms(v[m][0], v[m][1], top, half);
            const auto add = [&](const bf16x8 &p, const bf16x8 &s, float4_t &to) { to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p, s, to, 0, 0, 0); };
#pragma unroll
            for (int t = 0; t < MT; ++t) { add(a.high, b[t].high, high[C][m][t]); add(a.low, b[t].high, low[m][t]); }
#pragma unroll
            for (int t = 0; t < MT; ++t) add(a.mid, b[t].mid, low[m][t]);
#pragma unroll
            for (int t = 0; t < MT; ++t) add(a.high, b[t].low, low[m][t]);
#pragma unroll
            for (int t = 0; t < MT; ++t) add(a.mid, b[t].high, low[m][t]);
#pragma unroll
            for (int t = 0; t < MT; ++t) add(a.high, b[t].mid, low[m][t]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    request(0u);
    for (uint32_t step = 0; step < steps; step += 2u) {
        multiply(step, std::integral_constant<int, 0>{});
        if (step + 1u < steps) multiply(step + 1u, std::integral_constant<int, 1>{});
    }
    // a thread: four consecutive rows of a token (D[i = 4q .. 4q + 3][j = r])
    const uint32_t at = each_trip(tid), t = (at >> 6) % MT, m = (at >> 6) / MT, l = at & 63u, tok = tile_t * BT + 16u * t + (l & 15u), row = 4u * (l >> 4);      // (nothing of it in front of the first request)
    const bool has = at < (swiglu ? MR / 2u : MR) * MT * 64u && tok < ntok;
    static_assert(MR * MT * 64u <= 512u, "four outputs a thread");
    const auto meet = [&](auto part) {                     // the waves' sums in LDS
        __syncthreads();
#pragma unroll
        for (int mm = 0; mm < MR; ++mm)
#pragma unroll
            for (int tt = 0; tt < MT; ++tt) (&lds[0][0][0])[(wave * MR * MT + mm * MT + tt) * 64u + lane] = part(mm, tt);
        __syncthreads();
    };
    const auto products = [&](uint32_t mm) {
        double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const float4_t v = (&lds[0][0][0])[(k * MR * MT + mm * MT + t) * 64u + l];
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[i] += v[i];
        }
        return float4_t{(float)sum[0], (float)sum[1], (float)sum[2], (float)sum[3]};
    };
    // stores those of a thread's outputs that `which` names (a bit each) and whose products are finite or `last`; returns the rest
    const auto store = [&](uint32_t which, bool last) {
        float4_t y = products(m), u{};
        if (swiglu) u = products(m + MR / 2u);
        float *to = out + (uint64_t)tok * out_stride + block_row(m) + row;
        uint32_t now = 0u;
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            if ((fabsf(y[i]) <= 3.402823466e38f && fabsf(u[i]) <= 3.402823466e38f) || last) now |= which & (1u << i);
            if (swiglu) y[i] = (y[i] / (1.0f + expf(-y[i]))) * u[i];
        }
        if (swiglu && now == 15u) *reinterpret_cast<float4_t *>(to) = y;
        else {
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i)
                if (now >> i & 1u) to[i] = y[i];
        }
        which &= ~now;
        return which;
    };
    uint32_t which = 0u;                                   // outputs of this thread that are to be stored
    if (has) {
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) which |= swiglu || block_row(m) + row + i < all_rows ? 1u << i : 0u;
    }
    if (tid == 0u) again = 0u;
    meet([&](int mm, int tt) { return high[0][mm][tt] + high[1][mm][tt] + low[mm][tt]; });
    if (which) which = store(which, false);
    if (which) again = 1u;
    wave_lds_barrier();                                    // (not for the stores)
    if (!again) return;
    // the tile once more on the fp32 unit, for the others
    float4_t sum[MR][MT];
#pragma unroll
    for (int mm = 0; mm < MR; ++mm)
#pragma unroll
        for (int tt = 0; tt < MT; ++tt) sum[mm][tt] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    request(0u);
    for (uint32_t step = 0; step < steps; ++step) {
        float4_t v[NB][2];
        fetched(step, v);
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k)
#pragma unroll
            for (int mm = 0; mm < MR; ++mm)
#pragma unroll
                for (int tt = 0; tt < MT; ++tt)
                    sum[mm][tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[mm][k / 4u][k % 4u], v[MR + tt][k / 4u][k % 4u], sum[mm][tt], 0, 0, 0);
    }
    meet([&](int mm, int tt) { return sum[mm][tt]; });
    if (which) store(which, true);
}

// The tile that costs least: rounds of the device (256 compute units) times what a round of workgroups of it takes, 18, 10 and 7 us for 2048
// columns of 64 x 32, 32 x 32 and 32 x 16 outputs (gate/up of 512 tokens 20 / 22.5 / 29 us, of 77 tokens 16.7 / 11.1 / 8.2, down of 77 tokens, 512
// columns, 7.1 / 5.0 / 5.5, router of 512 tokens 18.5 / 12.7 / 16).
template <F32Kind KIND>
hipError_t f32_tiles(const float *w, const float *extra_row, const float *x, uint32_t ntok, uint32_t K, uint32_t n_rows, float *out, uint32_t out_stride, void *xh, void *xl,
                     int *xexp, hipStream_t s) {
    if (!ntok || !K || K % 256u || !n_rows || !w || !x || !out || (KIND == F32_SWIGLU && n_rows % 128u)) return hipErrorInvalidValue;
    const uint32_t all_rows = n_rows + (extra_row && !xh ? 1u : 0u);
    static constexpr struct { uint32_t br, bt, round; } kTiles[3] = {{64u, 32u, 18u}, {32u, 32u, 10u}, {32u, 16u, 7u}};
    uint64_t n[3], best = ~0ull;
    int pick = 0;
    for (int i = 0; i < 3; ++i) {
        n[i] = (uint64_t)((all_rows + kTiles[i].br - 1u) / kTiles[i].br) * ((ntok + kTiles[i].bt - 1u) / kTiles[i].bt);
        const uint64_t cost = (n[i] + 255u) / 256u * kTiles[i].round;
        if (cost < best) { best = cost; pick = i; }
    }
    const uint32_t split_wgs = xh ? (ntok + 7u) / 8u : 0u;      // (behind the tiles)
    if (n[pick] + split_wgs > 0x7fffffffull) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)n[pick] + split_wgs), block(512u);
    _Float16 *h = static_cast<_Float16 *>(xh), *l = static_cast<_Float16 *>(xl);
    if (pick == 0) REDHIP_LAUNCH((f32_tiles_kernel<4, 2, KIND>), grid, block, 0, s, w, extra_row, x, out, out_stride, h, l, xexp, K, n_rows, ntok, Beside<KIND>{});
    else if (pick == 1) REDHIP_LAUNCH((f32_tiles_kernel<2, 2, KIND>), grid, block, 0, s, w, extra_row, x, out, out_stride, h, l, xexp, K, n_rows, ntok, Beside<KIND>{});
    else REDHIP_LAUNCH((f32_tiles_kernel<2, 1, KIND>), grid, block, 0, s, w, extra_row, x, out, out_stride, h, l, xexp, K, n_rows, ntok, Beside<KIND>{});
    return hipGetLastError();
}

// out[tok][row] = W[row] . x[tok] for an f32 matrix W [n_rows][K] and a chunk of activations x [ntok][K]; extra_row (optional) is one more
// row behind the matrix; xh / xl / xexp (optional): also write the fp16 halves of x
hipError_t launch_f32_tiles(const float *w, const float *extra_row, const float *x, uint32_t ntok, uint32_t K, uint32_t n_rows, float *out,
                            uint32_t out_stride, void *xh, void *xl, int *xexp, hipStream_t s) {
    return f32_tiles<F32_PLAIN>(w, extra_row, x, ntok, K, n_rows, out, out_stride, xh, xl, xexp, s);
}
// act[tok][c] = silu(W[c] . x[tok]) * (W[ffn + c] . x[tok])
hipError_t launch_f32_swiglu_tiles(const float *w, const float *x, uint32_t ntok, uint32_t K, uint32_t ffn, float *act, hipStream_t s) {
    return f32_tiles<F32_SWIGLU>(w, nullptr, x, ntok, K, 2u * ffn, act, ffn, nullptr, nullptr, nullptr, s);
}

hipError_t launch_router_f32_tiles(const float *w, const float *gate_inp, const float *x, uint32_t ntok, uint32_t hidden, uint32_t n_expert,
                                   float *logits, void *xh, void *xl, int *xexp, hipStream_t s) {
    return f32_tiles<F32_PLAIN>(w, gate_inp, x, ntok, hidden, n_expert, logits, n_expert + 1u, xh, xl, xexp, s);
}

// The shared expert of a small chunk as part of the launch that precedes its routing: act = silu(gate) * up as launch_f32_swiglu_tiles, the router's
// logits (none with n_expert = 0: then the gate's factor goes to scalar) and the fp16 halves of the activations, in tiles of 32 x 16. Where they are less
// than two rounds of the device the launch takes hardly longer than the router alone, while the same products on a stream of their own cost the chunk
// 15 us, most of it the fork and the join. Us per layer on the other stream -> here: IQ1_M, 2048 x 512, 28 tokens 113 -> 100, 77 tokens 164 -> 155;
// IQ3_S down 33 tokens 129 -> 115, 100 tokens (349 workgroups) 177 -> 175, IQ2_XS 160 tokens (500) 226 -> 227; 2048 x 768, 120 tokens (431) 152 -> 145;
// 1024 x 256, 33 tokens 64 -> 51, 300 tokens (399) 77 -> 72. With the routing given the launch that splits the activations is shorter than a router:
// IQ1_M 30 tokens 104 -> 97, IQ2_XS 110 tokens (238 workgroups) 199 -> 197, IQ3_S 200 tokens (441) 202 -> 206.
bool front_tiles_fit(uint32_t ntok, uint32_t ffn, uint32_t n_expert) {
    return ffn % 64u == 0u && (uint64_t)(ffn / 16u + (n_expert + 31u) / 32u) * ((ntok + 15u) / 16u) + (ntok + 7u) / 8u <= (n_expert ? 448u : 256u);
}
hipError_t launch_front_tiles(const float *gate_up, const float *router, const float *gate_inp, const float *x, uint32_t ntok, uint32_t hidden, uint32_t ffn, uint32_t n_expert,
                              float *act, float *logits, float *scalar, void *xh, void *xl, int *xexp, hipStream_t s) {
    if (!ntok || !hidden || hidden % 256u || !front_tiles_fit(ntok, ffn, n_expert) || !gate_up || !gate_inp || !x || !act || !xh || !xl || !xexp || (n_expert ? !router || !logits : !scalar))
        return hipErrorInvalidValue;
    const dim3 grid((ffn / 16u + (n_expert + 31u) / 32u) * ((ntok + 15u) / 16u) + (ntok + 7u) / 8u);
    REDHIP_LAUNCH((f32_tiles_kernel<2, 1, F32_BOTH>), grid, dim3(512), 0, s, gate_up, gate_inp, x, act, ffn, static_cast<_Float16 *>(xh), static_cast<_Float16 *>(xl), xexp, hidden,
                  2u * ffn, ntok, Beside<F32_BOTH>{{router, logits, n_expert ? nullptr : scalar, n_expert, n_expert + 1u}});
    return hipGetLastError();
}

}  // namespace redhip
