// What a chunk of tokens (prefill) needs beside its tile kernels (redhip_tiles.hip): the tile lists, the tile-major copies of the experts'
// matrices, and dense f32 products on the fp32 matrix units (router logits, the shared expert of mixed layouts).
#include <hip/hip_runtime.h>

#include "redhip_mfma.h"

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

// out[tok][row] = W[row] . x[tok] for an f32 matrix W (a router, the dense shared expert of mixed layouts) and a chunk of activations, on
// v_mfma_f32_16x16x4_f32 (full fp32 multiply-add). A workgroup owns BR = 16 MR WR rows x BT = 16 MT WT tokens; a wave MR blocks of 16 rows times
// MT of 16 tokens, and half of k: the waves come in two sets, one for the even slices of 64 k, one for the odd ones, whose sums meet in LDS at
// the end. Both operands pass through LDS (SLICE k of either half per round, double-buffered, the next two rounds in registers). Lane
// (r = l % 16, q = l / 16) reads four consecutive k of row r and of token r and feeds them to four MFMAs (A[i = r][k = q], B[k = q][j = r],
// D[i = 4q .. 4q + 3][j = r]; the order of k does not matter as long as both operands agree).
// What bounds it: the matrix pipe where a tile is large (64 x 64: 16 bytes of L2 per clock and compute unit; tiles of 32 x 32 for every size
// needed 32, and waited for them), the number of workgroups where a chunk is small. So the tile is chosen by the launch (f32_tile_choice).
// The order in which an output's products are added is the same for every tile. The matrix unit rounds with every product, so the dense
// products leave it after 32 columns and are added up in double: of a shared expert's 2048-column rows 0.9e-7 is lost instead of 3.5e-7 (and of
// the output of an IQ1_M layer 1.6e-7 instead of 6e-7). A router keeps two plain chains: nothing but the selection hangs on its last bits.
// SWIGLU: W holds gate rows, then as many up rows; two row blocks beside each other are the gate and the up rows of 16 columns, and out gets
// silu(gate) * up of them: no pass of its own over the products.
// Launches with xh get workgroups behind the tiles that write the fp16 halves of the activations (a wave per token, split_token) and multiply them
// with gate_inp, if there is one, as row n_rows; without xh the tiles have it as a further row.

__device__ __forceinline__ void split_token(const float *gate_inp, const float *x, float *logits, uint32_t out_stride, _Float16 *xh, _Float16 *xl, int *xexp, uint32_t H,
                                            uint32_t E, uint32_t tok, uint32_t lane) {
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
                if (gate_inp) logits[(uint64_t)tok * out_stride + E] = gate;
            }
}

template <int MR, int MT, uint32_t WR, uint32_t WT, uint32_t SLICE, bool SWIGLU, bool ROUTER>
__global__ __launch_bounds__(128 * WR * WT) void f32_tiles_kernel(const float *w, const float *gate_inp, const float *x, float *out, uint32_t out_stride, _Float16 *xh,
                                                                  _Float16 *xl, int *xexp, uint32_t K, uint32_t n_rows, uint32_t ntok) {
    constexpr uint32_t BR = 16u * MR * WR, BT = 16u * MT * WT, T = 128u * WR * WT, P = SLICE / 4u, D = T / (2u * P), NW = BR / D, NX = BT / D;      // P pieces of 16 bytes per row, D rows per pass of the threads
    __shared__ __attribute__((aligned(16))) float lds[2][2][BR + BT][SLICE + 4u];      // [buffer][k half][W rows, then tokens]
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t all_rows = n_rows + (gate_inp && !xh ? 1u : 0u), row_tiles = (all_rows + BR - 1u) / BR, tok_tiles = (ntok + BT - 1u) / BT, n_tile = row_tiles * tok_tiles;
    if (blockIdx.x >= n_tile) {
        const uint32_t tok = T / 64u * (blockIdx.x - n_tile) + wave;
        if (tok < ntok) split_token(gate_inp, x, out, out_stride, xh, xl, xexp, K, n_rows, tok, lane);
        return;
    }
    // Workgroups are dealt to the eight XCDs in turn, each with its own L2: workgroup i lands on XCD i % 8. The tiles of one XCD form a
    // compact block of the tile grid (a quarter of the row tiles x half of the token tiles), so that an XCD fetches a quarter of the
    // matrix and half of the activations instead of all of both. (A different dealing order would only cost this locality.)
    uint32_t tile_r = blockIdx.x % row_tiles, tile_t = blockIdx.x / row_tiles;
    if (row_tiles % 4u == 0u && tok_tiles % 2u == 0u) {
        const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3, br = row_tiles / 4u, bt = tok_tiles / 2u;
        tile_r = (xcd & 3u) * br + slot % br;
        tile_t = (xcd >> 2) * bt + slot / br;
    }
    // staging: thread t moves the 16 bytes t % P of k half (t / P) % 2 of rows t / 2P, t / 2P + D, ..; rows and tokens beyond the last repeat
    // another and are not stored. (LDS rows of SLICE + 4 floats: the sixteen lanes of a 16-byte read pass hit different banks)
    const uint32_t scol = 4u * (tid % P), kh = (tid / P) & 1u, srow = tid / (2u * P);
    const auto source = [&](uint32_t n) -> const float * {      // (n < NW: matrix rows, then tokens)
        const uint32_t l = srow + n * D;
        if (n >= NW) return x + (uint64_t)min(tile_t * BT + l - BR, ntok - 1u) * K + kh * 64u + scol;
        const uint32_t row = SWIGLU ? ((l >> 4) & 1u) * (n_rows / 2u) + tile_r * (BR / 2u) + (l >> 5) * 16u + (l & 15u) : tile_r * BR + l;
        return (row < n_rows ? w + (uint64_t)row * K : gate_inp ? gate_inp : w) + kh * 64u + scol;
    };
    constexpr uint32_t N = NW + NX;
    static_assert(N >= 3u && N <= 6u && NW * D == BR && NX * D == BT && (SLICE == 32u || SLICE == 64u), "16-byte pieces per thread and round");
    const float *src0 = source(0u), *src1 = source(1u), *src2 = source(2u), *src3 = source(3u < N ? 3u : 0u), *src4 = source(4u < N ? 4u : 0u), *src5 = source(5u < N ? 5u : 0u);
    const uint32_t n_round = K / (2u * SLICE);             // even: K is a multiple of 256
    struct Staged { float4_t v0, v1, v2, v3, v4, v5; };    // (as an array, or of float4 objects, these end up in scratch memory)
    const auto request = [&](Staged &st, uint32_t rd) {    // (the last rounds request themselves again: no branch around the loads)
        const uint32_t at = SLICE == 64u ? rd * 128u : (rd >> 1) * 128u + (rd & 1u) * 32u;
        st.v0 = *reinterpret_cast<const float4_t *>(src0 + at);
        st.v1 = *reinterpret_cast<const float4_t *>(src1 + at);
        st.v2 = *reinterpret_cast<const float4_t *>(src2 + at);
        if constexpr (N > 3u) st.v3 = *reinterpret_cast<const float4_t *>(src3 + at);
        if constexpr (N > 4u) st.v4 = *reinterpret_cast<const float4_t *>(src4 + at);
        if constexpr (N > 5u) st.v5 = *reinterpret_cast<const float4_t *>(src5 + at);
    };
    const auto place = [&](const Staged &st, uint32_t buf) {      // (tokens follow the rows)
        *reinterpret_cast<float4_t *>(&lds[buf][kh][srow][scol]) = st.v0;
        *reinterpret_cast<float4_t *>(&lds[buf][kh][srow + D][scol]) = st.v1;
        *reinterpret_cast<float4_t *>(&lds[buf][kh][srow + 2u * D][scol]) = st.v2;
        if constexpr (N > 3u) *reinterpret_cast<float4_t *>(&lds[buf][kh][srow + 3u * D][scol]) = st.v3;
        if constexpr (N > 4u) *reinterpret_cast<float4_t *>(&lds[buf][kh][srow + 4u * D][scol]) = st.v4;
        if constexpr (N > 5u) *reinterpret_cast<float4_t *>(&lds[buf][kh][srow + 5u * D][scol]) = st.v5;
    };
    const uint32_t mh = wave / (WR * WT), block = wave % (WR * WT), wr = block % WR, wt = block / WR;
    constexpr int CH = ROUTER ? 2 : 1;
    float4_t acc[MR][MT][CH];
    double total[MR][MT][4];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int c = 0; c < CH; ++c) acc[m][t][c] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 4; ++i) total[m][t][i] = 0.0;
        }
    const auto multiply = [&](uint32_t buf) {
#pragma unroll
        for (uint32_t u = 0; u < SLICE / 16u; ++u) {
            float4 a[MR], b[MT];
#pragma unroll
            for (int m = 0; m < MR; ++m) a[m] = *reinterpret_cast<const float4 *>(&lds[buf][mh][16u * (MR * wr + m) + r][16u * u + 4u * q]);
#pragma unroll
            for (int t = 0; t < MT; ++t) b[t] = *reinterpret_cast<const float4 *>(&lds[buf][mh][BR + 16u * (MT * wt + t) + r][16u * u + 4u * q]);
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int m = 0; m < MR; ++m)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[m][t][k % CH] = __builtin_amdgcn_mfma_f32_16x16x4f32(k == 0 ? a[m].x : k == 1 ? a[m].y : k == 2 ? a[m].z : a[m].w,
                                                                                k == 0 ? b[t].x : k == 1 ? b[t].y : k == 2 ? b[t].z : b[t].w, acc[m][t][k % CH], 0, 0, 0);
            if constexpr (!ROUTER)
                if (u & 1u) {
#pragma unroll
                    for (int m = 0; m < MR; ++m)
#pragma unroll
                        for (int t = 0; t < MT; ++t) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) total[m][t][i] += acc[m][t][0][i];
                            acc[m][t][0] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
                        }
                }
        }
    };
    Staged s0, s1;
    request(s0, 0u);
    request(s1, 1u);
    for (uint32_t rd = 0; rd < n_round; rd += 2u) {
        place(s0, 0u);
        __syncthreads();                                   // round rd is in place; the readers of the other buffer (round rd - 1) are past their barrier
        request(s0, rd + 2u < n_round ? rd + 2u : rd);
        multiply(0u);
        place(s1, 1u);
        __syncthreads();
        request(s1, rd + 3u < n_round ? rd + 3u : rd + 1u);
        multiply(1u);
    }
    float4_t sum[MR][MT];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[m][t][i] = ROUTER ? acc[m][t][0][i] + acc[m][t][CH - 1][i] : (float)total[m][t][i];
        }
    // the odd slices' sums go through LDS to the waves that hold the even ones; SWIGLU with one row block per wave: then the up products to
    // the wave of their gate rows
    float4_t *meet = reinterpret_cast<float4_t *>(&lds[0][0][0][0]);
    static_assert(sizeof(lds) >= (size_t)WR * WT * MR * MT * 64u * 16u, "the sums fit the staging buffers");
    const auto at = [&](uint32_t b, int m, int t) { return ((b * MR + m) * MT + t) * 64u + lane; };
    __syncthreads();
    if (mh == 1u) {
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int t = 0; t < MT; ++t) meet[at(block, m, t)] = sum[m][t];
    }
    __syncthreads();
    if (mh == 0u) {
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int t = 0; t < MT; ++t) sum[m][t] += meet[at(block, m, t)];
    }
    if constexpr (SWIGLU && MR == 1) {
        if (mh == 0u && (wr & 1u)) {
#pragma unroll
            for (int t = 0; t < MT; ++t) meet[at(block, 0, t)] = sum[0][t];      // (its own place: nobody else reads it before)
        }
        __syncthreads();
    }
    if (mh == 1u || (SWIGLU && MR == 1 && (wr & 1u))) return;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const uint32_t tok = tile_t * BT + 16u * (MT * wt + t) + r;
        if (tok >= ntok) continue;
        if constexpr (SWIGLU) {
            float4_t y;
            const float4_t g = sum[0][t], u = MR == 1 ? meet[at(block + 1u, 0, t)] : sum[MR - 1][t];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = (g[i] / (1.0f + expf(-g[i]))) * u[i];
            *reinterpret_cast<float4_t *>(out + (uint64_t)tok * out_stride + tile_r * (BR / 2u) + 16u * (MR == 1 ? wr / 2u : wr) + 4u * q) = y;
        } else {
#pragma unroll
            for (int m = 0; m < MR; ++m)
#pragma unroll
                for (uint32_t i = 0; i < 4u; ++i) {
                    const uint32_t row = tile_r * BR + 16u * (MR * wr + m) + 4u * q + i;
                    if (row < all_rows) out[(uint64_t)tok * out_stride + row] = sum[m][t][i];
                }
        }
    }
}

// The largest tile that costs no more rounds of the device (256 compute units, workgroups of equal length) than a quarter above the best
// tile: large tiles read less, small ones fill the device when a chunk has few outputs.
template <bool SWIGLU, bool ROUTER>
hipError_t f32_tiles(const float *w, const float *extra_row, const float *x, uint32_t ntok, uint32_t K, uint32_t n_rows, float *out, uint32_t out_stride, void *xh, void *xl,
                     int *xexp, hipStream_t s) {
    if (!ntok || !K || K % 256u || !n_rows || !w || !x || !out || (SWIGLU && n_rows % 128u)) return hipErrorInvalidValue;
    const uint32_t all_rows = n_rows + (extra_row && !xh ? 1u : 0u);
    static constexpr struct { uint32_t br, bt; } kTiles[4] = {{64u, 64u}, {64u, 32u}, {32u, 32u}, {32u, 16u}};
    uint64_t n[4], cost[4], best = ~0ull;
    for (int i = 0; i < 4; ++i) {
        n[i] = (uint64_t)((all_rows + kTiles[i].br - 1u) / kTiles[i].br) * ((ntok + kTiles[i].bt - 1u) / kTiles[i].bt);
        cost[i] = (n[i] + 255u) / 256u * (kTiles[i].br * kTiles[i].bt);
        if (cost[i] < best) best = cost[i];
    }
    int pick = 0;
    while (4u * cost[pick] > 5u * best) ++pick;
    const uint32_t waves = pick < 3 ? 8u : 4u, split_wgs = xh ? (ntok + waves - 1u) / waves : 0u;      // (behind the tiles)
    if (n[pick] + split_wgs > 0x7fffffffull) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)n[pick] + split_wgs), block(64u * waves);
    _Float16 *h = static_cast<_Float16 *>(xh), *l = static_cast<_Float16 *>(xl);
    if (pick == 0) REDHIP_LAUNCH((f32_tiles_kernel<2, 2, 2u, 2u, 32u, SWIGLU, ROUTER>), grid, block, 0, s, w, extra_row, x, out, out_stride, h, l, xexp, K, n_rows, ntok);
    else if (pick == 1) REDHIP_LAUNCH((f32_tiles_kernel<2, 1, 2u, 2u, 32u, SWIGLU, ROUTER>), grid, block, 0, s, w, extra_row, x, out, out_stride, h, l, xexp, K, n_rows, ntok);
    else if (pick == 2) REDHIP_LAUNCH((f32_tiles_kernel<1, 1, 2u, 2u, 64u, SWIGLU, ROUTER>), grid, block, 0, s, w, extra_row, x, out, out_stride, h, l, xexp, K, n_rows, ntok);
    else REDHIP_LAUNCH((f32_tiles_kernel<1, 1, 2u, 1u, 64u, SWIGLU, ROUTER>), grid, block, 0, s, w, extra_row, x, out, out_stride, h, l, xexp, K, n_rows, ntok);
    return hipGetLastError();
}

// out[tok][row] = W[row] . x[tok] for an f32 matrix W [n_rows][K] and a chunk of activations x [ntok][K]; extra_row (optional) is one more
// row behind the matrix; xh / xl / xexp (optional): also write the fp16 halves of x
hipError_t launch_f32_tiles(const float *w, const float *extra_row, const float *x, uint32_t ntok, uint32_t K, uint32_t n_rows, float *out,
                            uint32_t out_stride, void *xh, void *xl, int *xexp, hipStream_t s) {
    return f32_tiles<false, false>(w, extra_row, x, ntok, K, n_rows, out, out_stride, xh, xl, xexp, s);
}
// act[tok][c] = silu(W[c] . x[tok]) * (W[ffn + c] . x[tok])
hipError_t launch_f32_swiglu_tiles(const float *w, const float *x, uint32_t ntok, uint32_t K, uint32_t ffn, float *act, hipStream_t s) {
    return f32_tiles<true, false>(w, nullptr, x, ntok, K, 2u * ffn, act, ffn, nullptr, nullptr, nullptr, s);
}

hipError_t launch_router_f32_tiles(const float *w, const float *gate_inp, const float *x, uint32_t ntok, uint32_t hidden, uint32_t n_expert,
                                   float *logits, void *xh, void *xl, int *xexp, hipStream_t s) {
    return f32_tiles<false, true>(w, gate_inp, x, ntok, hidden, n_expert, logits, n_expert + 1u, xh, xl, xexp, s);
}

}  // namespace redhip
