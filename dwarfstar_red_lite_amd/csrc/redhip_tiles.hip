// Chunks of tokens (prefill): the (token, expert) pairs of one expert are cut into tiles of up to 32 pairs (build_tile_lists) and multiplied
// on v_mfma_f32_16x16x32_f16. Experts as raw GGUF rows (IQ2_XXS, IQ2_XS, IQ1_M, down also IQ3_S), as packed IQ2_XXS rows, or as tile-major
// copies of these formats (redhip_prefill.hip).
// Reference behaviour this replaces: native/redmetal_engine_prefill.m:1246-1330 (grouped GEMM over expert slices)
// with the arithmetic of native/redlite_native_reference.c:251-382.
//
// What bounds these kernels is the decode (every weight is decoded once per tile): 512 raw IQ2_XXS experts with ten pairs each keep the LDS busy
// 58 % of the gate/up launch (half of that conflicts of the table reads), the vector pipes 67 %, the matrix pipes 24 %, in waves that take
// turns. So the rows must cost nothing extra. Operand mapping (lane l, r = l % 16, q = l / 16): A[i = r][k = 8q .. 8q + 7] activations of pair r, B[k][j = r] weights
// of row r, D[i = 4q .. 4q + 3][j = r]: the lane's own row against four pairs. Which columns the instruction's k stand for is free as
// long as both operands agree: step s of a block of 256 columns takes columns 64 q + 8 s .. + 7 of it, so lane (r, q) decodes quarter q of
// its row's block and nothing else. Its fields are one 16-byte load (XS 4, IQ3_S 12 more bytes) that no other lane repeats, the four lanes
// of a row read 64 consecutive bytes, every bit position is a constant, and a scale (per 16 or 32 columns) is formed once for the
// entries that share it. (With step s = group s of the block, every lane of a row would load all of it: four times the requests.)
//
// K is cut into KP blocks of 256 columns, and NRT row tiles of 16 rows are in work beside each other (KP * NRT = 8; 6 with three
// blocks). A unit is two halves ("m") of 16 NRT rows: the gate and the up rows of 16 NRT FFN columns, or 32 NRT rows of a down matrix.
// A wave keeps the activations of its block for the whole tile in registers (fp16 halves hi + lo 2^-11, 22 significant bits of every value
// down to 2^-28 of the largest) and the rows of the next two units on their way; the blocks meet in LDS, one barrier per two units. Tiles of up to 16 pairs run sixteen waves, one half
// each (64 registers of activations, four waves per SIMD: the reads and the arithmetic of different waves overlap), tiles of 17 .. 32
// pairs eight waves with both halves and two sets of pairs per decoded weight, as a launch of their own. The SwiGLU activations go to
// the down kernel as f32, so work is cut at any unit, not at groups of columns that share an exponent; the down kernel splits them per
// pair and block when it loads them.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "redhip_quarter.h"

namespace redhip {

namespace {

constexpr uint32_t staged_nrt(uint32_t KP) { return KP == 3u ? 2u : 8u / KP; }
constexpr uint32_t staged_threads(int sets, uint32_t KP) { return 64u * KP * staged_nrt(KP) * (sets == 1 ? 2u : 1u); }

struct StagedArgs {
    const uint8_t *experts, *shared;       // first matrix of expert e at experts + e * stride, of the shared expert at `shared`
    uint64_t stride, mat_step;             // mat_step: gate/up, distance of the up matrix
    uint64_t d_off;                        // not raw rows: the block scales behind the quarters of a matrix (tile-major IQ2_XS: the scale bytes behind them)
    const uint32_t *pair_token, *tile_expert, *tile_pair0, *tile_n, *n_tiles;
    const _Float16 *xh, *xl;               // gate/up in: [ntok][K]
    const int *xexp;                       // [ntok]
    float *act;                            // [P + shared tokens][rows]: gate/up out; down in as [..][K]
    float *tmp, *sh_tmp;                   // down out: [P][rows] routed pairs, [ntok][rows] shared expert
    const int8_t *grid;                    // codebook of IQ2_XS / IQ1_M
    uint32_t rows, P, list_stride;
    uint32_t few;                          // wide tiles that are not worth a launch: fewer than this many
};

__device__ __forceinline__ void wave_lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Hides from the compiler that v is the same in every trip of a loop: what is cheap to form again from it must not be kept in registers
// (which the activations need) across the loop.
__device__ __forceinline__ uint32_t each_trip(uint32_t v) { asm volatile("" : "+v"(v)); return v; }

// What the units of a workgroup need to know of their tiles (gate/up: the pairs' tokens among it), fetched at the kernel's head by its
// first wave while the others build the tables; tiles beyond the first kTileInfos are looked up when they begin.
constexpr uint32_t kTileInfos = 32u;
struct TileInfo { uint64_t mat; uint32_t p0, n; };      // mat: distance of the expert's first matrix from StagedArgs::experts

// units u0 .. u1 - 1 (unit = tile * units per tile + unit of the tile) of a tile list; SETS sets of 16 pairs per tile
template <int SRC, bool DOWN, int SETS, uint32_t KP>
__device__ __forceinline__ void staged_units(const StagedArgs &a, const uint32_t *tile_expert, const uint32_t *tile_pair0, const uint32_t *tile_n, uint32_t u0,
                                             uint32_t u1, float *part, float *scales, TileInfo *tiles, uint32_t *tokens, uint8_t *entries, uint32_t *signs, const LaneTables &lt) {
    constexpr uint32_t NRT = staged_nrt(KP), WV = KP * NRT, T = staged_threads(SETS, KP), M = SETS == 1 ? 1u : 2u;      // M: halves per wave
    constexpr uint32_t K = 256u * KP, seg_rows = 16u * NRT, tile_bytes = 16u * KP * src_block<SRC>();
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), w8 = wave % WV, m_first = SETS == 1 ? wave / WV : 0u, kc = w8 % KP, rt = w8 / KP;
    const uint32_t upt = a.rows / ((DOWN ? 2u : 1u) * seg_rows);
    const auto matrix_of = [&](uint32_t tile) {
        const uint32_t e = tile_expert[tile];
        return e == kSharedTile ? (uint64_t)(a.shared - a.experts) : (uint64_t)e * a.stride;
    };
    // the lane's quarters of a unit, and what their d are made from
    struct Carried { Quarter v[M]; uint2 d[M]; };
    const auto request = [&](Carried &c, const uint8_t *mat, uint32_t j) {
#pragma unroll
        for (uint32_t m = 0; m < M; ++m) {
            const uint32_t half = m_first + m, row_tile = (DOWN ? 2u * j + half : j) * NRT + rt;
            const uint8_t *mm = mat + (DOWN ? 0u : half * a.mat_step), *ds = mm + a.d_off + row_tile * (KP * 32u);
            load_quarter<SRC, KP>(mm + (uint64_t)row_tile * tile_bytes, ds, fmt<SRC>() == F_XS ? mm + a.d_off + (uint64_t)a.rows * KP * 2u + row_tile * (KP * 128u) : nullptr, r, kc, q, c.v[m], c.d[m]);
        }
    };
    const uint32_t tile0 = u0 / upt, n_info = (u1 - 1u) / upt + 1u - tile0 < kTileInfos ? (u1 - 1u) / upt + 1u - tile0 : kTileInfos;
    const auto token_of = [&](uint32_t p0, uint32_t n, uint32_t i) {           // (pairs beyond the tile's n repeat its first one: their rows of the product are never stored)
        const uint32_t p = i < n ? p0 + i : p0;
        return p < a.P ? a.pair_token[p] : p - a.P;
    };
    if (tid < 64u) {
        if (tid < n_info) tiles[tid] = TileInfo{matrix_of(tile0 + tid), tile_pair0[tile0 + tid], tile_n[tile0 + tid]};
        if constexpr (!DOWN)
            for (uint32_t k = tid; k < n_info * 16u * SETS; k += 64u) tokens[k] = token_of(tile_pair0[tile0 + k / (16u * SETS)], tile_n[tile0 + k / (16u * SETS)], k % (16u * SETS));
    } else
        build_staged_tables<SRC, T - 64u>(entries, signs, tid - 64u, a.grid);
    __syncthreads();
    const auto uniform64 = [](uint64_t v) {
        return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v);
    };
    const auto info_of = [&](uint32_t tile) {
        if (tile - tile0 >= kTileInfos) return TileInfo{matrix_of(tile), tile_pair0[tile], tile_n[tile]};
        const TileInfo ti = tiles[tile - tile0];
        return TileInfo{uniform64(ti.mat), (uint32_t)__builtin_amdgcn_readfirstlane(ti.p0), (uint32_t)__builtin_amdgcn_readfirstlane(ti.n)};
    };
    // Precision. The matrix unit rounds a sum four times per instruction (once per eight products), so what a block's sum loses goes with the
    // length of its chain of instructions: the low halves have a chain of their own, and the high ones one per kChain steps, added up in
    // f32 (in the registers, or where these are full in the LDS that takes the block's sum anyway). A chunk of normal rows comes out 1.9e-7
    // off (f32 multiplications: 2.1e-7); with one chain for everything it was 2.9e-7, in 3 .. 5 % less time. Packed rows (all-IQ2_XXS, ffn
    // above 512) take two steps per chain: 1.75e-7 instead of 1.9e-7, 5 % of the time.
    constexpr uint32_t kChain = layout<SRC>() == L_ROWS ? 2u : 4u;
    constexpr bool kSumInLds = SRC == S_IQ3 || (SETS == 2 && layout<SRC>() == L_ROWS);
    // Units on their way: two, one where the registers hold no second (a spill to scratch memory would be counted among the loads that the
    // waits count). Codebook wide tiles with two and the sums in the LDS instead: 2048 tokens IQ1_M 743 against 732 us, IQ2_XS 793 against 782.
    constexpr uint32_t kCarried = SRC == S_IQ3 || (SETS == 2 && fmt<SRC>() != F_XXS) ? 1u : 2u;
    H8 xa[SETS][8], xb[SETS][8];
    // Powers of two that the products of a pair are multiplied with. Down: of this wave's block. Gate/up: of the token, so the sums over the
    // blocks take them; a tile's stand in row tile % 4: a tile has two units or more, so the first wave is at most two tiles ahead of the
    // one that still adds sums up.
    float *pair_scale = scales + (DOWN ? wave * 16u * SETS : 0u);
    const auto load_tile = [&](uint32_t tile, uint32_t p0, uint32_t n) {
#pragma unroll
        for (uint32_t s = 0; s < (uint32_t)SETS; ++s) {
            __builtin_amdgcn_sched_barrier(0);             // one set at a time: both at once do not fit the registers
            const uint32_t l = each_trip(lane), lq = l >> 4, i = 16u * s + (l & 15u);
            float scale;
            if constexpr (!DOWN) {
                const uint32_t tok = tile - tile0 < kTileInfos ? tokens[(tile - tile0) * 16u * SETS + i] : token_of(p0, n, i);
                scale = format_scale<SRC>() * exp2i(a.xexp[tok]);
                const uint64_t base = (uint64_t)tok * K + 256u * kc;
                const _Float16 *hp = a.xh + base, *lp = a.xl + base;
#pragma unroll
                for (uint32_t g = 0; g < 8u; ++g) {
                    xa[s][g].u = *reinterpret_cast<const uint4 *>(hp + step_column<SRC>(g, lq));
                    xb[s][g].u = *reinterpret_cast<const uint4 *>(lp + step_column<SRC>(g, lq));
                }
                if (s + 1u == (uint32_t)SETS) __builtin_amdgcn_s_waitcnt(0x0f70);      // vmcnt(0): waited for here, once per tile, not (by count) where the loop uses them
            } else {
                // f32 activations of pair p, columns of this wave's K part: one exponent for them, then the fp16 halves
                const float *src = a.act + (uint64_t)(i < n ? p0 + i : p0) * K + 256u * kc;
                float amax = 0.0f;
#pragma unroll
                for (uint32_t g = 0; g < 8u; ++g) {
                    const float4 v0 = *reinterpret_cast<const float4 *>(src + step_column<SRC>(g, lq)), v1 = *reinterpret_cast<const float4 *>(src + step_column<SRC>(g, lq) + 4u);
                    xa[s][g].u = __builtin_bit_cast(uint4, v0);
                    xb[s][g].u = __builtin_bit_cast(uint4, v1);
                }
#pragma unroll
                for (uint32_t g = 0; g < 8u; ++g) {
                    const float4 v0 = __builtin_bit_cast(float4, xa[s][g].u), v1 = __builtin_bit_cast(float4, xb[s][g].u);
                    amax = fmaxf(amax, fmaxf(fmaxf(fmaxf(fabsf(v0.x), fabsf(v0.y)), fmaxf(fabsf(v0.z), fabsf(v0.w))), fmaxf(fmaxf(fabsf(v1.x), fabsf(v1.y)), fmaxf(fabsf(v1.z), fabsf(v1.w)))));
                }
                amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
                amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
                const int e = prescale_exp(amax);
                const float inv = exp2i(-e);
                scale = format_scale<SRC>() * exp2i(e);
#pragma unroll
                for (uint32_t g = 0; g < 8u; ++g) {
                    const float4 v0 = __builtin_bit_cast(float4, xa[s][g].u), v1 = __builtin_bit_cast(float4, xb[s][g].u);
                    const float f[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
                    H8 hi, lo;
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const float t = f[k] * inv;
                        const _Float16 h = (_Float16)t;
                        hi.e[k] = h;
                        lo.e[k] = (_Float16)split_rest(t, h);
                    }
                    // group by group (the compiler otherwise works on several at once and spills)
                    asm volatile("" : "+v"(hi.u.x), "+v"(hi.u.y), "+v"(hi.u.z), "+v"(hi.u.w), "+v"(lo.u.x), "+v"(lo.u.y), "+v"(lo.u.z), "+v"(lo.u.w));
                    xa[s][g].u = hi.u;
                    xb[s][g].u = lo.u;
                }
            }
            pair_scale[(DOWN ? 0u : (tile & 3u) * 16u * SETS) + i] = scale;      // (every lane and wave that has pair i writes the same)
        }
    };
    // partial sums of the waves: [row tile, K part][m][set][lane] float4
    constexpr uint32_t kWavePart = 2u * SETS * 256u, kPart = WV * kWavePart;      // (kPart: of a unit)
    struct Done { uint32_t tile, j, p0, n; };              // a unit whose partial sums are in LDS
    // The sums of UNITS units (w[0], and w[1] behind it). No wave and no lane may skip a store: the loads of the next units are in flight
    // behind it, and the compiler, which waits for them by counting memory operations in order, can count only what every path issues
    // (with a branch around it, every unit waited for the newest of its loads). Pairs beyond a tile's n fall out of the buffer's range.
    const auto tile_buffer = [&](float *base, uint32_t n) { return __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)(n * a.rows * 4u), 0x00027000); };
    using Sum = std::conditional_t<(KP > 2u), double, float>;      // (a row's partial sums are added here one after the other)
    const auto reduce = [&](auto units, const Done *w, const float *pt) {
        constexpr uint32_t UNITS = decltype(units)::value;
        const uint32_t t = each_trip(tid);
        if constexpr (DOWN) {
            // V consecutive floats (pairs of one row) per thread; threads beyond the last repeat it
            constexpr uint32_t V = SETS == 1 ? 2u : 4u, PB = 256u / V, N = PB * SETS * 2u * NRT;
#pragma unroll
            for (uint32_t un = 0; un < UNITS; ++un) {
                const bool routed = w[un].p0 < a.P;        // (a tile is routed or shared as a whole)
                const auto buf = tile_buffer((routed ? a.tmp + (uint64_t)w[un].p0 * a.rows : a.sh_tmp + (uint64_t)(w[un].p0 - a.P) * a.rows), w[un].n);
#pragma unroll
                for (uint32_t base = 0; base < N; base += T) {
                    const uint32_t it = N % T ? min(base + t, N - 1u) : base + t;
                    const uint32_t at = (it & (PB - 1u)) * V, b = it / PB, set = b & (SETS - 1u), m = (b / SETS) & 1u, slot = b / (2u * SETS);
                    const float *src = pt + un * kPart + slot * KP * kWavePart + (m * SETS + set) * 256u + at;
                    Sum s[V];
#pragma unroll
                    for (uint32_t v = 0; v < V; ++v) s[v] = src[v];
#pragma unroll
                    for (uint32_t k = 1; k < KP; ++k)
#pragma unroll
                        for (uint32_t v = 0; v < V; ++v) s[v] += src[k * kWavePart + v];
                    const uint32_t i = 16u * set + 4u * (at >> 6) + (at & 3u), off = 4u * (i * a.rows + w[un].j * 2u * seg_rows + m * seg_rows + 16u * slot + ((at >> 2) & 15u));
#pragma unroll
                    for (uint32_t v = 0; v < V; ++v) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((float)s[v]), buf, off + 4u * v * a.rows, 0, 0);
                }
            }
        } else {
            // (pair, column) elements; L lanes of a wave (halves of it) share one where there are fewer elements than threads
            constexpr uint32_t N = 256u * SETS * NRT * UNITS, L = N < T ? T / N : 1u;
            static_assert(L <= 4u && KP % L == 0u, "K parts per lane");
#pragma unroll
            for (uint32_t base = 0; base < N; base += T) {
                const uint32_t ln = t & 63u, e = base + (L == 1u ? t : (t >> 6) * (64u / L) + (ln & (64u / L - 1u))), k0 = L == 1u ? 0u : (ln / (64u / L)) * (KP / L);
                const uint32_t at = e & 255u, b = (e >> 8) % (SETS * NRT), un = (e >> 8) / (SETS * NRT), set = b & (SETS - 1u), slot = b / SETS;
                const float *src = pt + un * kPart + (slot * KP + k0) * kWavePart + set * 256u + at;
                Sum s0 = src[0], s1 = src[SETS * 256u];
#pragma unroll
                for (uint32_t k = 1; k < KP / L; ++k) {
                    s0 += src[k * kWavePart];
                    s1 += src[k * kWavePart + SETS * 256u];
                }
                if constexpr (L >= 2u) { s0 += __shfl_xor(s0, 32, 64); s1 += __shfl_xor(s1, 32, 64); }
                if constexpr (L == 4u) { s0 += __shfl_xor(s0, 16, 64); s1 += __shfl_xor(s1, 16, 64); }
                // (the wave's elements are of one unit)
                const uint32_t uw = UNITS == 1u ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(un);
                const Done d = uw ? w[UNITS - 1u] : w[0];
                const auto buf = tile_buffer(a.act + (uint64_t)d.p0 * a.rows, d.n);
                const uint32_t i = 16u * set + 4u * (at >> 6) + (at & 3u);
                const float scale = pair_scale[(d.tile & 3u) * 16u * SETS + i], g = (float)s0 * scale, up = (float)s1 * scale;
                // (of the lanes that share an element the first stores; the others' offset lies beyond every buffer)
                const uint32_t off = k0 == 0u ? 4u * (i * a.rows + d.j * seg_rows + 16u * slot + ((at >> 2) & 15u)) : 0x7fffffffu;
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint((g / (1.0f + expf(-g))) * up), buf, off, 0, 0);
            }
        }
    };
    uint32_t tile = tile0, j = u0 % upt, ftile = tile0, fj = j, fleft = u1 - u0;      // f..: the unit to be requested next
    TileInfo cur = info_of(tile);
    uint64_t fmat = cur.mat;
    const auto request_next = [&](Carried &c) {            // (the last units fetch theirs again: registers filled under a condition would be live all around the loop)
        request(c, a.experts + fmat, fj);
        if (fleft <= 1u) return;
        --fleft;
        if (++fj == upt) { fj = 0u; fmat = info_of(++ftile).mat; }
    };
    // multiplies the unit whose rows are in c into partial sums at pt and requests the unit two after it in their place
    const auto unit = [&](uint32_t u, Carried &c, float *pt) {
        float4_t acc[M][SETS], low[M][SETS], sum[M][SETS];
        float d[M];
#pragma unroll
        for (uint32_t m = 0; m < M; ++m) {
            d[m] = quarter_d<SRC>(c.d[m]);
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s) acc[m][s] = low[m][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
        float *mine = pt + w8 * kWavePart + m_first * SETS * 256u + 4u * lane;
        Entry e[M];
        half2_t f[M];
#pragma unroll
        for (uint32_t m = 0; m < M; ++m) e[m] = fetch_entry<SRC>(c.v[m], 0u, lt);
#pragma unroll
        for (uint32_t s8 = 0; s8 < 8u; ++s8) {
            // table reads run a step ahead of the products (two steps ahead takes five registers more per row and was no quicker)
            __builtin_amdgcn_sched_barrier(0);
            half8_t w[M];
#pragma unroll
            for (uint32_t m = 0; m < M; ++m) {
                if constexpr (steps_per_scale<SRC>() != 0u) { if (s8 % steps_per_scale<SRC>() == 0u) f[m] = step_scale<SRC>(c.v[m], s8); }
                w[m] = finish_entry<SRC>(e[m], f[m]);
                if (s8 < 7u) e[m] = fetch_entry<SRC>(c.v[m], s8 + 1u, lt);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (s8 == 6u) request_next(c);                 // (the quarters' last use is behind)
            if (s8 && s8 % kChain == 0u) {                 // put the sums so far aside
#pragma unroll
                for (uint32_t m = 0; m < M; ++m)
#pragma unroll
                    for (uint32_t s = 0; s < (uint32_t)SETS; ++s) {
                        float4_t &so_far = kSumInLds ? *reinterpret_cast<float4_t *>(mine + (m * SETS + s) * 256u) : sum[m][s];
                        so_far = s8 == kChain ? acc[m][s] : so_far + acc[m][s];
                        acc[m][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    }
            }
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s)
#pragma unroll
                for (uint32_t m = 0; m < M; ++m) acc[m][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[s][s8].v, w[m], acc[m][s], 0, 0, 0);
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s)
#pragma unroll
                for (uint32_t m = 0; m < M; ++m) low[m][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[s][s8].v, w[m], low[m][s], 0, 0, 0);
        }
#pragma unroll
        for (uint32_t m = 0; m < M; ++m)
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s) {
                float4_t *at = reinterpret_cast<float4_t *>(mine + (m * SETS + s) * 256u);
                if constexpr (kSumInLds) sum[m][s] = *at;
                float4_t factor = {d[m], d[m], d[m], d[m]};
                if constexpr (DOWN) factor *= *reinterpret_cast<const float4_t *>(pair_scale + 16u * s + 4u * q);
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[m][s][t] = fmaf(low[m][s][t], 4.8828125e-4f, sum[m][s][t] + acc[m][s][t]) * factor[t];
                *at = acc[m][s];
            }
        const Done done{tile, j, cur.p0, cur.n};
        if (++j == upt && u + 1u < u1) { j = 0u; cur = info_of(++tile); load_tile(tile, cur.p0, cur.n); }
        return done;
    };
    Carried c[kCarried];
#pragma unroll
    for (uint32_t k = 0; k < kCarried; ++k) request_next(c[k]);
    load_tile(tile, cur.p0, cur.n);
    // narrow: two units per barrier, four buffers of partial sums; wide: one, two buffers (as large). A buffer is written again two
    // barriers after its sums were complete; whoever adds them has passed one in between.
    constexpr std::integral_constant<uint32_t, 1u> one{};
    constexpr std::integral_constant<uint32_t, 2u> two{};
    uint32_t u = u0;
    float *pt = part;
    for (; u + 1u < u1; u += 2u) {
        Done w[2];
        w[0] = unit(u, c[0], pt);
        if constexpr (SETS == 2) {
            wave_lds_barrier();
            reduce(one, w, pt);
        }
        w[1] = unit(u + 1u, c[kCarried - 1u], pt + kPart);
        wave_lds_barrier();
        if constexpr (SETS == 2) reduce(one, w + 1, pt + kPart);
        else {
            reduce(two, w, pt);
            pt = pt == part ? part + 2u * kPart : part;
        }
    }
    if (u < u1) {
        const Done w = unit(u, c[0], pt);
        wave_lds_barrier();
        reduce(one, &w, pt);
    }
}

// SETS 1: the narrow tiles (list 2) of a chunk, SETS 2: the wide ones (list 1). Persistent workgroups, each with an equal run of the units.
// A launch that finds few wide tiles leaves them: the narrow one then takes every pair in tiles of 16 (list 0). Two launches where one would
// do cost 10 to 20 us (tables, the first tiles' activations, compute units without a unit at both ends); a wide tile saves a second decoding
// of its rows, which goes with their weights. So the line is a number of weights in wide tiles: 220 million for gate/up, 230 million for
// IQ2_XXS down rows, 145 million for the other down formats. Both ways measured on chunks of evenly routed tokens, 128 and 512 experts with
// 12 to 40 pairs on average, 1024 x 256 to 2048 x 768; what was even: gate/up 130 to 240 million on all-IQ2_XXS layers, 300 to 450 on the
// others, down 118 to 230 IQ2_XXS, 125 to 170 the others. 221 wide tiles of 2048 x 512 (464 / 232 million, IQ2_XS): 260 + 133 us with
// them, 263 + 154 without; 97 (203 / 102): 105 + 69 against 99 + 54. On mixed layouts the shared expert's products run beside gate/up and
// finish sooner beside two launches: a layer of 112 wide tiles of 2048 x 512 (235 million) takes 332 us with them, 340 without, one of 195
// of 1024 x 512 (205) 191 against 183, so these share the all-IQ2_XXS line. Packed IQ2_XXS down rows (ffn above 512) lost 20 us with 57 to
// 139 wide tiles alike and have none.
template <int SRC, bool DOWN> constexpr bool has_wide() { return !(DOWN && layout<SRC>() == L_ROWS); }
template <int SRC, bool DOWN> uint32_t few_wide(uint32_t rows, uint32_t K) {
    return !has_wide<SRC, DOWN>() ? ~0u : (DOWN ? fmt<SRC>() == F_XXS ? 230000000u : 145000000u : 110000000u) / (rows * K) + 1u;
}
template <int SRC, bool DOWN, int SETS, uint32_t KP>
__global__ __launch_bounds__(staged_threads(SETS, KP)) void staged_tiles_kernel(StagedArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t entries[kEntryBytes];   // static: table reads take immediate offsets
    __shared__ __attribute__((aligned(16))) uint32_t signs[sign_bytes<SRC>() / 4u + 4u];
    __shared__ __attribute__((aligned(16))) float part[4u * KP * staged_nrt(KP) * 2u * 256u];
    const uint32_t n0 = a.n_tiles[0], n1 = a.n_tiles[1], n2 = a.n_tiles[2];      // (one trip)
    const bool few = n1 < a.few;
    if (SETS == 2 && few) return;
    const uint32_t tid = threadIdx.x, l = SETS == 2 ? 1u : few ? 0u : 2u, off = l * a.list_stride;
    const uint32_t units = (SETS == 2 ? n1 : few ? n0 : n2) * (a.rows / ((DOWN ? 32u : 16u) * staged_nrt(KP)));
    // workgroups are dealt round-robin over the eight XCDs: neighbouring runs (which share tiles) go to one XCD's L2
    const uint32_t G = gridDim.x, at = G % 8u == 0u ? (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u : blockIdx.x;
    const uint32_t u0 = (uint32_t)((uint64_t)at * units / G), u1 = (uint32_t)((uint64_t)(at + 1u) * units / G);
    if (u0 >= u1) return;
    __shared__ TileInfo tiles[kTileInfos];
    __shared__ uint32_t tokens[DOWN ? 1u : kTileInfos * 16u * SETS];
    __shared__ __attribute__((aligned(16))) float scales[(DOWN ? staged_threads(SETS, KP) / 64u : 4u) * 16u * SETS];
    const LaneTables lt{entries + (fmt<SRC>() == F_XS ? (tid & 7u) * 16u : fmt<SRC>() == F_M ? (tid & 1u) * 16u : 0u),
                        reinterpret_cast<const uint8_t *>(signs) + (is_iq3<SRC>() ? (tid & 3u) * 4u : fmt<SRC>() == F_M ? 0u : (tid & 15u) * 4u)};
    staged_units<SRC, DOWN, SETS, KP>(a, a.tile_expert + off, a.tile_pair0 + off, a.tile_n + off, u0, u1, part, scales, tiles, tokens, entries, signs, lt);
}

template <int SRC, bool DOWN, int SETS, uint32_t KP>
hipError_t launch_staged_list(const StagedArgs &a, uint32_t grid, hipStream_t s) {
    REDHIP_LAUNCH((staged_tiles_kernel<SRC, DOWN, SETS, KP>), dim3(grid), dim3(staged_threads(SETS, KP)), 0, s, a);
    return hipGetLastError();
}
// wide: wide tiles that the chunk is expected to have
template <int SRC, bool DOWN, uint32_t KP>
hipError_t launch_staged_lists(StagedArgs a, uint32_t grid, uint32_t wide, hipStream_t s) {
    a.few = few_wide<SRC, DOWN>(a.rows, 256u * KP);
    hipError_t e = hipSuccess;
    if (wide < a.few) a.few = ~0u;                         // (without a wide launch the narrow one takes everything)
    if constexpr (has_wide<SRC, DOWN>()) {
        if (a.few != ~0u) e = launch_staged_list<SRC, DOWN, 2, KP>(a, grid, s);
    }
    return e == hipSuccess ? launch_staged_list<SRC, DOWN, 1, KP>(a, grid, s) : e;
}
template <int SRC>
hipError_t staged_gateup(const StagedArgs &a, uint32_t hidden, uint32_t grid, uint32_t wide, hipStream_t s) {
    return hidden == 512u    ? launch_staged_lists<SRC, false, 2>(a, grid, wide, s)
           : hidden == 1024u ? launch_staged_lists<SRC, false, 4>(a, grid, wide, s)
                             : launch_staged_lists<SRC, false, 8>(a, grid, wide, s);
}
template <int SRC>
hipError_t staged_down(const StagedArgs &a, uint32_t ffn, uint32_t grid, uint32_t wide, hipStream_t s) {
    if (ffn == 256u) return launch_staged_lists<SRC, true, 1>(a, grid, wide, s);
    if (ffn == 512u) return launch_staged_lists<SRC, true, 2>(a, grid, wide, s);
    if constexpr (layout<SRC>() == L_TILED) return hipErrorInvalidValue;      // (tile-major copies are made for ffn <= 512)
    else return ffn == 768u ? launch_staged_lists<SRC, true, 3>(a, grid, wide, s) : launch_staged_lists<SRC, true, 4>(a, grid, wide, s);
}

int staged_src(uint32_t type, RowLayout lay) {
    if (lay == RowLayout::rows) return type == T_IQ2_XXS ? S_ROWS_XXS : -1;
    if (lay == RowLayout::tiled) return type == T_IQ2_XXS ? S_TILED_XXS : type == T_IQ2_XS ? S_TILED_XS : type == T_IQ1_M ? S_TILED_M : type == T_IQ3_S ? S_TILED_IQ3 : -1;
    return type == T_IQ2_XXS ? S_XXS : type == T_IQ2_XS ? S_XS : type == T_IQ1_M ? S_M : type == T_IQ3_S ? S_IQ3 : -1;
}

StagedArgs staged_args(const StagedMatrices &m, const StagedChunk &c, uint32_t K, uint32_t rows) {
    const int src = staged_src(m.type, m.layout);
    StagedArgs a{};
    a.experts = static_cast<const uint8_t *>(m.experts);
    a.shared = static_cast<const uint8_t *>(m.shared);
    a.stride = m.stride;
    a.mat_step = m.up_delta;
    a.d_off = src == S_TILED_IQ3 ? (uint64_t)rows * (K / 32u) * 16u : (uint64_t)rows * (K / 32u) * 8u;
    a.pair_token = c.pair_token;
    a.tile_expert = c.tl.tile_expert; a.tile_pair0 = c.tl.tile_pair0; a.tile_n = c.tl.tile_n; a.n_tiles = c.tl.n_tiles;
    a.list_stride = c.tl.list_stride;
    a.grid = m.grid;
    a.rows = rows;
    a.P = c.ntok * c.top_k;
    return a;
}
// persistent workgroups, one per compute unit; fewer where a chunk cannot have as many units as that
uint32_t staged_grid(const StagedChunk &c) {
    const uint32_t bound = 4u * prefill_tile_bound(c.ntok, c.top_k, c.n_expert);
    return bound < 256u ? bound : 256u;
}
// Wide tiles that a chunk will have: counted by the caller, or guessed. A launch that finds too few costs 5 us, and a wide tile has 17 pairs or
// more, so a chunk has at most pairs / 17 of them: 0.37 of that with Zipf-popular experts (512 and 1024 tokens, top 10 of 512), next to none
// at ten evenly routed pairs per expert, one for nearly every expert from 23 pairs on, a further one per 32 from 42 on.
uint32_t staged_wide(const StagedChunk &c) {
    if (c.wide_tiles != kWideUnknown) return c.wide_tiles;
    const uint32_t pairs = c.ntok * c.top_k, E = c.n_expert, popular = pairs / (kPrefillTile + 1u) * 2u / 5u, first = pairs > 10u * E ? (pairs - 10u * E) / 13u : 0u;
    const uint32_t routed = (first < E ? first : E) + (pairs > 42u * E ? (pairs - 42u * E) / kPrefillWideTile : 0u);
    return (routed < popular ? popular : routed) + c.tl.shared_ntok / kPrefillWideTile;
}

}  // namespace

bool staged_gateup_supported(uint32_t type, RowLayout lay, uint32_t hidden, uint32_t ffn) {
    const int src = staged_src(type, lay);
    return src >= 0 && type != T_IQ3_S && (hidden == 512u || hidden == 1024u || hidden == 2048u) && ffn && ffn % 128u == 0u;
}
// one block of 256 columns per wave: two to eight of them (hidden), one to four (ffn)
bool staged_down_supported(uint32_t type, RowLayout lay, uint32_t hidden, uint32_t ffn) {
    return staged_src(type, lay) >= 0 && hidden && hidden % 256u == 0u && (ffn == 256u || ffn == 512u || (lay != RowLayout::tiled && (ffn == 768u || ffn == 1024u)));
}

hipError_t launch_staged_gateup(const StagedMatrices &m, const StagedChunk &c, const void *xh, const void *xl, const int *xexp, float *act, uint32_t hidden, uint32_t ffn,
                                hipStream_t s) {
    if (!staged_gateup_supported(m.type, m.layout, hidden, ffn) || !c.ntok || (c.tl.shared_ntok && !m.shared)) return hipErrorInvalidValue;
    StagedArgs a = staged_args(m, c, hidden, ffn);
    a.xh = static_cast<const _Float16 *>(xh);
    a.xl = static_cast<const _Float16 *>(xl);
    a.xexp = xexp;
    a.act = act;
    const uint32_t grid = staged_grid(c);
    const uint32_t wide = staged_wide(c);
    prof_set_stage(ST_PREFILL_GATEUP);
    switch (staged_src(m.type, m.layout)) {
        case S_XXS: return staged_gateup<S_XXS>(a, hidden, grid, wide, s);
        case S_XS: return staged_gateup<S_XS>(a, hidden, grid, wide, s);
        case S_M: return staged_gateup<S_M>(a, hidden, grid, wide, s);
        case S_ROWS_XXS: return staged_gateup<S_ROWS_XXS>(a, hidden, grid, wide, s);
        case S_TILED_XXS: return staged_gateup<S_TILED_XXS>(a, hidden, grid, wide, s);
        case S_TILED_XS: return staged_gateup<S_TILED_XS>(a, hidden, grid, wide, s);
        case S_TILED_M: return staged_gateup<S_TILED_M>(a, hidden, grid, wide, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_staged_down(const StagedMatrices &m, const StagedChunk &c, const float *act, float *tmp, float *sh_tmp, uint32_t hidden, uint32_t ffn, hipStream_t s) {
    if (!staged_down_supported(m.type, m.layout, hidden, ffn) || !c.ntok || (c.tl.shared_ntok && (!m.shared || !sh_tmp))) return hipErrorInvalidValue;
    StagedArgs a = staged_args(m, c, ffn, hidden);
    a.act = const_cast<float *>(act);
    a.tmp = tmp;
    a.sh_tmp = sh_tmp;
    const uint32_t grid = staged_grid(c);
    const uint32_t wide = staged_wide(c);
    prof_set_stage(ST_PREFILL_DOWN);
    switch (staged_src(m.type, m.layout)) {
        case S_XXS: return staged_down<S_XXS>(a, ffn, grid, wide, s);
        case S_XS: return staged_down<S_XS>(a, ffn, grid, wide, s);
        case S_M: return staged_down<S_M>(a, ffn, grid, wide, s);
        case S_IQ3: return staged_down<S_IQ3>(a, ffn, grid, wide, s);
        case S_ROWS_XXS: return staged_down<S_ROWS_XXS>(a, ffn, grid, wide, s);
        case S_TILED_XXS: return staged_down<S_TILED_XXS>(a, ffn, grid, wide, s);
        case S_TILED_XS: return staged_down<S_TILED_XS>(a, ffn, grid, wide, s);
        case S_TILED_M: return staged_down<S_TILED_M>(a, ffn, grid, wide, s);
        case S_TILED_IQ3: return staged_down<S_TILED_IQ3>(a, ffn, grid, wide, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace redhip
