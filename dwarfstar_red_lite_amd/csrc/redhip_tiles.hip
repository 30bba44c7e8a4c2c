// Chunks of tokens (prefill): the (token, expert) pairs of one expert are cut into tiles of up to 32 pairs (build_tile_lists) and multiplied
// on v_mfma_f32_16x16x32_f16. Experts as raw GGUF rows (IQ2_XXS, IQ2_XS, IQ1_M, down also IQ3_S), as packed IQ2_XXS rows, or as tile-major
// copies of these formats (redhip_prefill.hip).
// Reference behaviour this replaces: native/redmetal_engine_prefill.m:1246-1330 (grouped GEMM over expert slices)
// with the arithmetic of native/redlite_native_reference.c:251-382.
//
// What bounds these kernels is the decode: every weight is decoded once per tile, eight of them for about ten vector instructions and a table read
// of 12 LDS cycles (conflicts of random entries), beside which the matrix instructions take 8 issue cycles each. So the rows must cost nothing
// extra. Operand mapping (lane l, r = l % 16, q = l / 16): A[i = r][k = 8q .. 8q + 7] activations of pair r, B[k][j = r] weights
// of row r, D[i = 4q .. 4q + 3][j = r]: the lane's own row against four pairs. Which columns the instruction's k stand for is free as
// long as both operands agree: step s of a block of 256 columns takes columns 64 q + 8 s .. + 7 of it, so lane (r, q) decodes quarter q of
// its row's block and nothing else. Its fields are one 16-byte load (XS 4, IQ3_S 12 more bytes) that no other lane repeats, the four lanes
// of a row read 64 consecutive bytes, every bit position is a constant, and a scale (per 16 or 32 columns) is formed once for the
// entries that share it. (With step s = group s of the block, every lane of a row would load all of it: four times the requests.)
//
// K is cut into KP blocks of 256 columns. The activations are fp16 halves hi + lo 2^-11 (22 significant bits of every value down to 2^-28 of the
// largest). A tile's 16 pairs times 2048 columns fill a quarter of the vector registers, so gate/up keeps them there, split over the waves by
// columns, and adds the waves' sums up in LDS; the 512 columns of a down tile fit the LDS, so there every wave has whole rows and nothing
// is added up (with whole rows and the activations of 2048 columns passing through LDS block by block, gate/up took 171 instead of 144 us).
// The SwiGLU activations go to the down kernel as f32, so work is cut at any unit, not at groups of columns that share an exponent.
// 512 raw IQ2_XXS experts of 2048 x 512 with ten pairs each: gate/up 130 us (small tiles as full ones 144; sixteen waves of one block, and the decode on full
// instruction rate only: 166), down 74 (83; 99, activations in registers too); 77 tokens of IQ1_M layers 70 + 40 (96 + 48; 112 + 68).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "redhip_quarter.h"

namespace redhip {

namespace {

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

// exchange of two registers' halves between lanes that differ in bit 4 (16) or 5 (32)
__device__ __forceinline__ void swap16(uint32_t &a, uint32_t &b) { const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false); a = r[0]; b = r[1]; }
__device__ __forceinline__ void swap32(uint32_t &a, uint32_t &b) { const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false); a = r[0]; b = r[1]; }
__device__ __forceinline__ void swap16(uint4 &a, uint4 &b) { swap16(a.x, b.x); swap16(a.y, b.y); swap16(a.z, b.z); swap16(a.w, b.w); }
__device__ __forceinline__ void swap32(uint4 &a, uint4 &b) { swap32(a.x, b.x); swap32(a.y, b.y); swap32(a.z, b.z); swap32(a.w, b.w); }

// What a workgroup needs to know of its tiles, fetched for up to kTileInfos of them at a time.
constexpr uint32_t kTileInfos = 32u;
struct TileInfo { uint64_t mat; uint32_t p0, n; };      // mat: distance of the expert's first matrix from StagedArgs::experts
struct TileList { const uint32_t *expert, *pair0, *n; };
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ TileInfo uniform_info(const TileInfo &t) { return TileInfo{((uint64_t)uni((uint32_t)(t.mat >> 32)) << 32) | uni((uint32_t)t.mat), uni(t.p0), uni(t.n)}; }
// the lane's quarter of block kc of row tile `row_tile` of a matrix of `rows` rows
template <int SRC, uint32_t KP>
__device__ __forceinline__ void request_quarter(const StagedArgs &a, const uint8_t *mat, uint32_t row_tile, uint32_t r, uint32_t kc, uint32_t q, Quarter &v, uint2 &d) {
    constexpr uint32_t tile_bytes = 16u * KP * src_block<SRC>();
    load_quarter<SRC, KP>(mat + (uint64_t)row_tile * tile_bytes, mat + a.d_off + row_tile * (KP * 32u),
                          fmt<SRC>() == F_XS ? mat + a.d_off + (uint64_t)a.rows * KP * 2u + row_tile * (KP * 128u) : nullptr, r, kc, q, v, d);
}
// g / (1 + exp(-g)). The exponent's product with log2(e) as two floats less its whole part, so that the result is as good as the exponential instruction; the
// quotient from the reciprocal and one step on what it leaves over, infinities and NaN as a division gives them. The reciprocal is of d / 4: that of 2^126
// and more, gates from -87.3 to -88.72, is below the normal floats, which the instruction does not give, while the quotient is not. In fewer instructions
// than expf and a division and as near to double: 0.370 units in the last place on average for gates of -20 .. 20 and 0.354 for -87 .. -20 (0.368 and 0.352);
// with 1 + the product's low part as a factor behind the exponential it was 0.435 and 0.511.
__device__ __forceinline__ float silu(float g) {
    const float c = __builtin_amdgcn_fmed3f(g, -128.0f, 128.0f), n = rintf(c * -1.44269502f), l = fmaf(c, -1.92596303e-8f, fmaf(c, -1.44269502f, -n));
    const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(l), (int)n), d = 1.0f + e, r = __builtin_amdgcn_rcpf(d * 0.25f) * 0.25f, x = g * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-x, d, g), r, x), d, g);
}
// rows `rows` long of the pairs of a tile: stores of pairs beyond n fall out of the range
// (base and n are the same in every lane; said again here, or the store would be in a loop over the lanes that have the same ones)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t pair_rows(float *rows_of_all, uint32_t p0, uint32_t n, uint32_t rows) {
    return __builtin_amdgcn_make_buffer_rsrc(rows_of_all + (uint64_t)uni(p0) * rows, 0, (int)(uni(n) * rows * 4u), 0x00027000);
}

// ---- gate/up ----
// SMALL: a tile of up to eight pairs, whose high and low halves are rows 0 .. 7 and 8 .. 15 of one operand: half the matrix instructions, half the
// activations. Tiles end with what is left of an expert's pairs, so these are a third (ten pairs an expert) to all (batches) of a chunk's: 77 tokens of
// IQ1_M layers 311 -> 286 us for two layers, a batch of 24 on IQ2_XXS 290 -> 271 for three, 512 tokens of a pool 204 -> 197.
// Eight waves. A wave keeps the activations of its columns for the whole tile in registers, as fp16 halves: of two blocks of 256 columns for
// sixteen pairs (SETS 1; it multiplies the gate or the up rows with them), of one block for 32 (SETS 2; both rows). PK such parts make the
// columns, NRT row tiles of 16 rows are in work beside each other: a unit is the gate and the up rows of 16 NRT FFN columns.
constexpr uint32_t kGateUpThreads = 512u;
template <int SETS, uint32_t KP> struct GateUp {
    static constexpr uint32_t PK = SETS == 1 ? KP / 2u : KP, NRT = SETS == 1 ? 4u / PK : 8u / PK, kUnits = SETS == 1 ? 4u : 1u;      // kUnits: between two barriers
    static constexpr uint32_t kSums = 512u * (uint32_t)SETS, kPart = NRT * PK * kSums;      // partial sums of a row tile's K part: [gate | up][set][256]; of a unit
};
template <int SRC, int SETS, uint32_t KP> struct GateUpLds {
    uint32_t signs[sign_bytes<SRC>() / 4u];              // the tables first: their reads then take the base as an immediate offset (16 bits)
    uint8_t entries[kEntryBytes];
    float part[2u * GateUp<SETS, KP>::kUnits * GateUp<SETS, KP>::kPart];
    TileInfo tiles[kTileInfos];
    float scales[kTileInfos * 16u * (uint32_t)SETS];     // powers of two that the sums of a pair are multiplied with
    uint32_t tokens[kTileInfos * 16u * (uint32_t)SETS];
};

// units u0 .. u1 - 1 (unit = tile * units per tile + unit of the tile) of a tile list
template <int SRC, int SETS, uint32_t KP, bool SHORT, bool SMALL>
__device__ __forceinline__ void gateup_units(const StagedArgs &a, const TileList &list, uint32_t u0, uint32_t u1, GateUpLds<SRC, SETS, KP> &lds, bool tables) {
    using G = GateUp<SETS, KP>;
    constexpr uint32_t PK = G::PK, NRT = G::NRT, K = 256u * KP, PAIRS = SMALL ? kPrefillSmallTile : 16u * SETS, T = kGateUpThreads, UB = G::kUnits;
    static_assert(!SMALL || SETS == 1, "");
    const uint32_t tid = each_trip(threadIdx.x), lane = tid & 63u, r = lane & 15u, q = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t kp = wave % PK, rt = (wave / PK) % NRT, up = wave / (PK * NRT);      // up: SETS 1, the wave has the up rows
    const uint32_t upt = a.rows / (16u * NRT), tile0 = u0 / upt, n_info = (u1 - 1u) / upt + 1u - tile0;
    // Everything that the first products wait for is on its way before the tables are built: the codebook, the run's tiles, their tokens, the first units'
    // rows, the first tile's activations, each behind what names it. (Fetched behind the tables and a barrier, the first products of a batch of 24
    // tokens began 13800 cycles into a launch of 89000.) Every thread requests the same number of loads, so that the waits can count them.
    TableSeeds<SRC, T> seeds;
    if (tables) seeds.request(tid, a.grid);
    constexpr uint32_t NI = (kTileInfos * PAIRS + T - 1u) / T;      // pairs of the run's tiles per thread
    struct { uint32_t e, p0, n, tok; int exp; } info[NI];
    const auto at_info = [&](uint32_t n) { return min(tid + n * T, n_info * PAIRS - 1u); };
#pragma unroll
    for (uint32_t n = 0; n < NI; ++n) {
        const uint32_t t = tile0 + at_info(n) / PAIRS;
        info[n].e = list.expert[t]; info[n].p0 = list.pair0[t]; info[n].n = list.n[t];
    }
    const auto mat_of = [&](uint32_t e) { return e == kSharedTile ? (uint64_t)(a.shared - a.experts) : (uint64_t)e * a.stride; };
    const uint32_t e0 = uni(list.expert[tile0]), e1 = uni(list.expert[tile0 + min(1u, n_info - 1u)]), first_p0 = uni(list.pair0[tile0]), first_n = uni(list.n[tile0]);
    const auto token_of = [&](uint32_t p0, uint32_t n, uint32_t i) {      // (pairs beyond the tile's n repeat its first one: their rows of the product are never stored)
        const uint32_t p = p0 + (i < n ? i : 0u), tok = a.pair_token[min(p, a.P - 1u)];
        return p < a.P ? tok : p - a.P;
    };
    const uint32_t pair = SMALL ? r & 7u : r;              // the lane's row of the activations
    uint32_t first_tok[SETS];
#pragma unroll
    for (uint32_t s = 0; s < (uint32_t)SETS; ++s) first_tok[s] = token_of(first_p0, first_n, 16u * s + pair);
#pragma unroll
    for (uint32_t n = 0; n < NI; ++n) info[n].tok = token_of(info[n].p0, info[n].n, at_info(n) % PAIRS);
    __builtin_amdgcn_sched_barrier(0);
    // the lane's two quarters of a unit (SETS 1: of the two blocks, SETS 2: of the gate and the up row), and what their d are made from
    struct Carried { Quarter v[2]; uint2 d[2]; };
    const auto request = [&](Carried &c, uint64_t mat, uint32_t j) {
#pragma unroll
        for (uint32_t m = 0; m < 2u; ++m) {
            const uint8_t *mm = a.experts + mat + (SETS == 1 ? up : m) * a.mat_step;
            request_quarter<SRC, KP>(a, mm, j * NRT + rt, r, SETS == 1 ? 2u * kp + m : kp, q, c.v[m], c.d[m]);
        }
    };
    constexpr uint32_t kCarried = SETS == 2 && (fmt<SRC>() != F_XXS || layout<SRC>() == L_ROWS) ? 1u : 2u;      // units on their way: two where the registers hold them
    Carried c[kCarried];
    uint32_t tile = tile0, j = u0 % upt, ftile = tile0, fj = j, fleft = u1 - u0;      // f..: the unit to be requested next
    uint64_t fmat = mat_of(e0);
    request(c[0], fmat, fj);
    if constexpr (kCarried == 2u) {                        // (a tile has two units at least)
        if (fleft > 1u) {
            --fleft;
            if (++fj == upt) { fj = 0u; ++ftile; fmat = mat_of(e1); }
        }
        request(c[1], fmat, fj);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t n = 0; n < NI; ++n) info[n].exp = a.xexp[info[n].tok];
    __builtin_amdgcn_sched_barrier(0);
    // Precision. The matrix unit rounds a sum four times per instruction (once per eight products), so what a block's sum loses goes with the
    // length of its chain of instructions: the low halves have a chain of their own, and the high ones one per kChain steps, added up in f32.
    // (SHORT: of two steps.) The low halves go first into a result, so that it is rounded once for both. Of a chunk 1.82e-7 is lost so, 1.74e-7 with short
    // chains, in 1 to 2 % more time; batches of fewer tokens are slices, which lose 1.76e-7, so these have short ones and are no further off on the
    // tiles (IQ2_XXS, 2048 x 512, 24 tokens with the routing given; chains of one step lose more in the additions).
    constexpr uint32_t kChain = SHORT || layout<SRC>() == L_ROWS ? 2u : 4u;
    H8 xa[2][8], xb[SMALL ? 1 : 2][8];                     // SETS 1: [block], SETS 2: [set]; high and low halves (SMALL: both in xa)
    const float row_scale = SMALL && q >= 2u ? 4.8828125e-4f : 1.0f;      // of the lane's rows of the products
    const auto fetch_block = [&](uint32_t x, uint32_t tok) {
        const uint64_t base = (uint64_t)tok * K + 256u * (SETS == 1 ? 2u * kp + x : kp) + 8u * q;
        const _Float16 *hp = (SMALL && r >= 8u ? a.xl : a.xh) + base, *lp = a.xl + base;
        // four lanes of a pair take 64 bytes side by side; the exchange makes them each lane's own run
#pragma unroll
        for (uint32_t g = 0; g < 8u; ++g) {
            const uint32_t at = 8u * (16u * ((g >> 1) & 1u) + 8u * (g & 1u) + 4u * (g >> 2));
            xa[x][g].u = *reinterpret_cast<const uint4 *>(hp + at);
            if constexpr (!SMALL) xb[x][g].u = *reinterpret_cast<const uint4 *>(lp + at);
        }
        __builtin_amdgcn_sched_barrier(0);                 // one block at a time: the addresses of both do not fit the registers
    };
    const auto arrange_blocks = [&] {
#pragma unroll
        for (uint32_t x = 0; x < 2u; ++x) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t g = 0; g < 8u; g += 2u) { swap16(xa[x][g].u, xa[x][g + 1u].u); if constexpr (!SMALL) swap16(xb[x][g].u, xb[x][g + 1u].u); }
#pragma unroll
            for (uint32_t g = 0; g < 8u; ++g) if (!(g & 2u)) { swap32(xa[x][g].u, xa[x][g + 2u].u); if constexpr (!SMALL) swap32(xb[x][g].u, xb[x][g + 2u].u); }
        }
    };
    const auto load_tile = [&](uint32_t tile) {
#pragma unroll
        for (uint32_t x = 0; x < 2u; ++x) {
            __builtin_amdgcn_sched_barrier(0);
            fetch_block(x, lds.tokens[(tile - tile0) * PAIRS + (SETS == 1 ? 0u : 16u * x) + (each_trip(threadIdx.x) & (SMALL ? 7u : 15u))]);
        }
        arrange_blocks();
    };
    const auto fill_lds = [&] {
        if (tables) seeds.store(lds.entries, lds.signs, tid);
#pragma unroll
        for (uint32_t n = 0; n < NI; ++n) {
            const uint32_t k = at_info(n);                 // (surplus threads repeat the last)
            lds.tokens[k] = info[n].tok;
            lds.scales[k] = format_scale<SRC>() * exp2i(info[n].exp);
            if (k % PAIRS == 0u) lds.tiles[k / PAIRS] = TileInfo{mat_of(info[n].e), info[n].p0, info[n].n};
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (SETS == 2) fill_lds();                   // (the registers do not hold the seeds beside the activations)
#pragma unroll
    for (uint32_t x = 0; x < 2u; ++x) fetch_block(x, first_tok[SETS == 1 ? 0u : x]);
    if constexpr (SETS == 1) fill_lds();
    wave_lds_barrier();
    const LaneTables lt = lane_tables<SRC>(lds.entries, lds.signs, tid);
    arrange_blocks();
    // The sums of UNITS units, the first of them number fj of tile ft, and their SwiGLU. No wave and no lane may skip a store: the loads of the next units are in flight in front of it, and the
    // compiler, which waits for them by counting memory operations in order, can count only what every path issues.
    // (What is done for every output is counted here too: a thread's outputs are the same place of different units, so their pair, its distance in `act` and
    // its scale are found once, and the tile stands in scalar registers.)
    TileInfo here{fmat, first_p0, first_n};                // the tile of the unit that is multiplied
    const auto reduce = [&](auto units, const TileInfo &of, uint32_t ft, uint32_t fj, const float *pt) {
        constexpr uint32_t UNITS = decltype(units)::value, OUT = 16u * (SMALL ? 8u : 16u), N = OUT * SETS * NRT * UNITS;      // OUT: a row tile's outputs, of sixteen pairs or of eight
        const uint32_t at = each_trip(threadIdx.x) % OUT, pair0 = 4u * (at >> 6) + (at & 3u), out_at = 4u * (pair0 * a.rows + ((at >> 2) & 15u));
#pragma unroll
        for (uint32_t base = 0; base < N; base += T) {
            const uint32_t b = uni(((base + threadIdx.x) % N) / OUT), un = b / (SETS * NRT), set = b % SETS, slot = (b / SETS) % NRT;      // (surplus threads repeat others' outputs)
            const float *src = pt + un * G::kPart + slot * PK * G::kSums + set * 256u + at;
            constexpr uint32_t PARTS = SMALL ? 2u * PK : PK;      // SMALL: the sums over high and over low halves apart
            using Sum = std::conditional_t<(PARTS > 1u), double, float>;      // (a row's parts are added here)
            Sum g[PARTS], u[PARTS];
#pragma unroll
            for (uint32_t k = 0; k < PARTS; ++k) {
                const uint32_t off = (k % PK) * G::kSums + (k / PK) * OUT;
                g[k] = src[off];
                u[k] = src[off + SETS * 256u];
            }
            uint32_t dt = ft - tile0, dj = fj + un;
            TileInfo d = of;
            if (dj >= upt) {
                while (dj >= upt) { dj -= upt; ++dt; }
                d = uniform_info(lds.tiles[dt]);
            }
            const float scale = lds.scales[dt * PAIRS + 16u * set + pair0];
#pragma unroll
            for (uint32_t n = PARTS / 2u; n; n /= 2u)
#pragma unroll
                for (uint32_t k = 0; k < n; ++k) { g[k] += g[k + n]; u[k] += u[k + n]; }
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(silu((float)g[0] * scale) * ((float)u[0] * scale)), pair_rows(a.act, d.p0, d.n, a.rows),
                                                  out_at + 64u * set * a.rows, 4u * (dj * 16u * NRT + 16u * slot), 0);
        }
    };
    const auto request_rows = [&](Carried &c) { request(c, fmat, fj); };
    const auto advance = [&] {                             // (the last units fetch theirs again: registers filled under a condition would be live all around the loop)
        if (fleft <= 1u) return;
        --fleft;
        if (++fj == upt) { fj = 0u; fmat = uniform_info(lds.tiles[++ftile - tile0]).mat; }
    };
    // multiplies the unit whose rows are in c into partial sums at pt and requests the unit two after it in their place
    const auto unit = [&](uint32_t u, Carried &c, float *pt) {
        float4_t acc[2][SETS], low[2][SETS], sum[2][SETS];
        float d[2];
        Entry e[2];
        half2_t f[2];
#pragma unroll
        for (uint32_t m = 0; m < 2u; ++m) {
            d[m] = quarter_d<SRC>(c.d[m]);
            if constexpr (SMALL) d[m] *= row_scale;
            e[m] = fetch_entry<SRC, 0u>(c.v[m], lt);
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s) acc[m][s] = low[m][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
        each_step([&](auto step) {
            constexpr uint32_t S = decltype(step)::value;
            // table reads run a step ahead of the products; who is behind goes first
            if constexpr (S % (SETS == 1 ? 4u : 2u) == 0u) __builtin_amdgcn_s_setprio(SETS == 1 ? 2 - (int)S / 2 : 3 - (int)S / 2);
            __builtin_amdgcn_sched_barrier(0);
            half8_t w[2];
#pragma unroll
            for (uint32_t m = 0; m < 2u; ++m) {
                if constexpr (steps_per_scale<SRC>() != 0u) { if constexpr (S % steps_per_scale<SRC>() == 0u) f[m] = step_scale<SRC, S>(c.v[m]); }
                w[m] = finish_entry<SRC>(e[m], f[m], lt);
                if constexpr (S < 7u) e[m] = fetch_entry<SRC, S + 1u>(c.v[m], lt);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (S == 6u) request_rows(c);        // (the quarters' last use is behind)
            if constexpr (S && S % kChain == 0u) {         // put the sums so far aside
#pragma unroll
                for (uint32_t m = 0; m < 2u; ++m)
#pragma unroll
                    for (uint32_t s = 0; s < (uint32_t)SETS; ++s) {
                        sum[m][s] = S == kChain ? acc[m][s] : sum[m][s] + acc[m][s];
                        acc[m][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    }
            }
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s)
#pragma unroll
                for (uint32_t m = 0; m < 2u; ++m) acc[m][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[SETS == 1 ? m : s][S].v, w[m], acc[m][s], 0, 0, 0);
            if constexpr (!SMALL) {
#pragma unroll
                for (uint32_t s = 0; s < (uint32_t)SETS; ++s)
#pragma unroll
                    for (uint32_t m = 0; m < 2u; ++m) low[m][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[SETS == 1 ? m : s][S].v, w[m], low[m][s], 0, 0, 0);
            }
        });
        float *mine = pt + (rt * PK + kp) * G::kSums + 4u * lane;
        if constexpr (SETS == 1) {
            float4_t &both = acc[0][0];                    // the two blocks
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if constexpr (SMALL) both[t] = fmaf(sum[1][0][t] + acc[1][0][t], d[1], (sum[0][0][t] + acc[0][0][t]) * d[0]);
                else {
                    const float l = fmaf(low[1][0][t], 4.8828125e-4f * d[1], low[0][0][t] * (4.8828125e-4f * d[0]));
                    both[t] = fmaf(sum[1][0][t] + acc[1][0][t], d[1], fmaf(sum[0][0][t] + acc[0][0][t], d[0], l));
                }
            }
            *reinterpret_cast<float4_t *>(mine + up * 256u) = both;
        } else {
#pragma unroll
            for (uint32_t m = 0; m < 2u; ++m)
#pragma unroll
                for (uint32_t s = 0; s < (uint32_t)SETS; ++s) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[m][s][t] = fmaf(sum[m][s][t] + acc[m][s][t], d[m], low[m][s][t] * (4.8828125e-4f * d[m]));
                    *reinterpret_cast<float4_t *>(mine + (m * SETS + s) * 256u) = acc[m][s];
                }
        }
        advance();
        if (++j == upt && u + 1u < u1) { j = 0u; here = uniform_info(lds.tiles[++tile - tile0]); load_tile(tile); }
    };
    advance();
    // A buffer of partial sums is written again two barriers after its sums were complete; whoever adds them has passed one in between.
    constexpr std::integral_constant<uint32_t, 1u> one{};
    constexpr std::integral_constant<uint32_t, UB> all{};
    uint32_t u = u0;
    float *pt = lds.part;
    const auto turn = [&] { pt = pt == lds.part ? lds.part + UB * G::kPart : lds.part; };
    for (; UB > 1u && u + UB <= u1; u += UB) {
        const uint32_t t = tile, j0 = j;
        const TileInfo of = here;
#pragma unroll
        for (uint32_t k = 0; k < UB; ++k) unit(u + k, c[k % kCarried], pt + k * G::kPart);
        wave_lds_barrier();
        reduce(all, of, t, j0, pt);
        turn();
    }
    const auto single = [&](Carried &cc) {
        const uint32_t t = tile, j0 = j;
        const TileInfo of = here;
        unit(u, cc, pt);
        wave_lds_barrier();
        reduce(one, of, t, j0, pt);
        turn();
        return ++u < u1;
    };
    if (u < u1) while (single(c[0]) && single(c[kCarried - 1u])) {}
}

// ---- down ----
// A tile's activations stand in LDS as fp16 halves, split once per tile: per panel (a block of 256 columns of sixteen pairs) and half the 16 bytes
// that lane l multiplies in step s at 1024 s + 16 l. A wave has whole rows, two row tiles beside each other, so it stores its sums from registers
// and waits for the others only where a tile begins. Narrow passes may take the end of one tile and the begin of the next where two fit the LDS.
constexpr uint32_t kPanel = 16384u;
constexpr uint32_t down_waves(int sets) { return sets == 1 ? 12u : 8u; }
template <int SETS, uint32_t KP> constexpr uint32_t down_tiles_a_pass() { return SETS == 1 && KP <= 2u ? 2u : 1u; }
template <int SRC, int SETS, uint32_t KP> struct DownLds {
    uint32_t signs[sign_bytes<SRC>() / 4u];
    uint8_t entries[small_tables<SRC>() ? small_entry_bytes<SRC>() : kEntryBytes];
    uint8_t x[(SETS == 2 ? 2u : down_tiles_a_pass<SETS, KP>()) * KP * kPanel];      // [tile % 2, or set][block]
    TileInfo tiles[kTileInfos];
    float scales[2u * KP * 16u * (uint32_t)SETS];        // [tile % 2][block][pair]: powers of two that the sums of a pair's block are multiplied with
};
// largest of the sixteen lanes of a row
__device__ __forceinline__ float row_max(float v) {
    const auto with = [](float x, auto ctrl) { return fmaxf(x, __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), decltype(ctrl)::value, 0xf, 0xf, false))); };
    v = with(v, std::integral_constant<int, 0xB1>{});      // quad_perm [1, 0, 3, 2], [2, 3, 0, 1]; row_ror 4, 8
    v = with(v, std::integral_constant<int, 0x4E>{});
    v = with(v, std::integral_constant<int, 0x124>{});
    return with(v, std::integral_constant<int, 0x128>{});
}

// Narrow tiles of up to two blocks: items i0 .. i1 - 1 of a tile list (item = tile * items per tile + item of the tile; an item: 32 rows, a wave's).
// Where a pass is of one tile: parts. A tile is `parts` passes, a run whole passes; cut by items, a run that crosses tiles has up to two passes more
// than its share, with waves idle in both (IQ3_S, 1024 x 768, 60 tiles: 46 us, now 35; 2048 x 768, 122 tiles: 58 -> 48). A part is a number of fours of
// items, one for each SIMD: 12 + 12 + 8 items are 2 % quicker than 11 + 11 + 10.
template <int SRC, int SETS, uint32_t KP, bool SMALL>
__device__ __forceinline__ void down_items(const StagedArgs &a, const TileList &list, uint32_t parts, uint32_t i0, uint32_t i1, DownLds<SRC, SETS, KP> &lds, bool tables) {
    constexpr uint32_t WV = down_waves(SETS), T = 64u * WV, PAIRS = SMALL ? kPrefillSmallTile : 16u * SETS, K = 256u * KP, kPassTiles = down_tiles_a_pass<SETS, KP>();
    constexpr uint32_t PANEL = SMALL ? kPanel / 2u : kPanel;
    static_assert(!SMALL || SETS == 1, "");
    const uint32_t tid = each_trip(threadIdx.x), lane = tid & 63u, r = lane & 15u, q = lane >> 4, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ipt = a.rows / 32u, tile0 = i0 / parts, n_info = (i1 - 1u) / parts + 1u - tile0, quads = ((ipt / 4u) << 16) / parts + 1u;      // quads: fours of items per part, 16 bits behind the point
    // A pass: an item per wave, of up to kPassTiles tiles
    struct Pass { uint32_t i, tile, j, n; };               // first item or part, its tile, the first item's number in the tile, items
    const auto pass_at = [&](uint32_t i, uint32_t tile, uint32_t at) {      // at: number of the item or part in the tile
        if constexpr (kPassTiles == 2u) return Pass{i, tile, at, (uint32_t)min(min(i1 - i, WV), 2u * ipt - at)};
        else {
            const uint32_t j = (at * quads >> 16) * 4u;
            return Pass{i, tile, j, ((at + 1u) * quads >> 16) * 4u - j};
        }
    };
    const auto last = [&](const Pass &p) { return p.i + (kPassTiles == 2u ? p.n : 1u) >= i1; };
    const auto following = [&](const Pass &p) {            // (behind the last pass: that one again)
        if (last(p)) return p;
        if constexpr (kPassTiles == 2u) {
            const uint32_t j = p.j + p.n, over = j >= ipt ? j >= 2u * ipt ? 2u : 1u : 0u;
            return pass_at(p.i + p.n, p.tile + over, j - over * ipt);
        } else {
            const uint32_t tile = p.tile + (p.j + p.n == ipt ? 1u : 0u);
            return pass_at(p.i + 1u, tile, p.i + 1u - tile * parts);
        }
    };
    const auto second = [&](const Pass &p) { return kPassTiles == 2u && p.j + min(wave, p.n - 1u) >= ipt ? 1u : 0u; };      // the wave's item is of the pass's second tile
    const auto last_tile = [&](const Pass &p) { return p.tile + (p.j + p.n > ipt ? 1u : 0u); };
    Pass p = pass_at(i0, tile0, i0 - tile0 * parts);
    // As in gate/up, what the first products wait for is on its way before the tables are built, and no thread skips a request: the codebook, the run's tiles, the
    // first pass's rows, the activations of the run's first two tiles.
    TableSeeds<SRC, T> seeds;
    SmallSeeds<SRC, T> small_seeds;
    if (tables) {
        if constexpr (small_tables<SRC>()) small_seeds.request(tid, a.grid);
        else seeds.request(tid, a.grid);
    }
    const uint32_t info_at = min(tid, n_info - 1u), info_e = list.expert[tile0 + info_at], info_p0 = list.pair0[tile0 + info_at], info_n = list.n[tile0 + info_at];
    const auto mat_of = [&](uint32_t e) { return e == kSharedTile ? (uint64_t)(a.shared - a.experts) : (uint64_t)e * a.stride; };
    const auto listed = [&](uint32_t t) { return TileInfo{mat_of(uni(list.expert[t])), uni(list.pair0[t]), uni(list.n[t])}; };
    const TileInfo first[2] = {listed(tile0), listed(tile0 + min(1u, n_info - 1u))};
    // the lane's quarters of a block of the wave's two row tiles, and what their d are made from
    struct Carried { Quarter v[2]; uint2 d[2]; };
    const auto request_block = [&](Carried &c, const Pass &p, uint64_t mat, uint32_t kb) {      // (a wave without an item requests the pass's last)
        const uint32_t item = p.j + min(wave, p.n - 1u) - second(p) * ipt;
#pragma unroll
        for (uint32_t m = 0; m < 2u; ++m) request_quarter<SRC, KP>(a, a.experts + mat, 2u * item + m, r, kb, q, c.v[m], c.d[m]);
    };
    Carried c[2];
    TileInfo now = first[second(p)];                       // the tile of the wave's item of pass p
    struct { Pass p; TileInfo info, before; uint32_t kb; } ahead{p, now, now, KP > 1u ? 2u % KP : 1u % KP};      // the block to be requested next; `before`: of the pass before it
    request_block(c[0], p, now.mat, 0u);
    if constexpr (KP > 1u) request_block(c[1], p, now.mat, 1u);
    __builtin_amdgcn_sched_barrier(0);
    // f32 activations of four pairs and a block per wave: one exponent for a pair's block, then the fp16 halves. Requested a tile ahead, kept in registers.
    constexpr uint32_t NS = (KP * PAIRS / 4u + WV - 1u) / WV;
    struct Staged { float4 v[NS][4]; };
    const auto fetch_tile = [&](Staged &st, uint32_t p0, uint32_t n) {
#pragma unroll
        for (uint32_t x = 0; x < NS; ++x) {
            const uint32_t w = min(wave + x * WV, KP * PAIRS / 4u - 1u), block = w / (PAIRS / 4u), i = (w % (PAIRS / 4u)) * 4u + q;
            const float *src = a.act + (uint64_t)(i < n ? p0 + i : p0) * K + 256u * block + 4u * r;
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) st.v[x][k] = *reinterpret_cast<const float4 *>(src + 64u * k);
        }
    };
    const auto put_tile = [&](const Staged &st, uint32_t tile) {
#pragma unroll
        for (uint32_t x = 0; x < NS; ++x) {
            const uint32_t w = wave + x * WV, block = w / (PAIRS / 4u), i = (w % (PAIRS / 4u)) * 4u + q;
            if (w >= KP * PAIRS / 4u) break;
            const float4 *v = st.v[x];
            float amax = 0.0f;
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[k].x), fabsf(v[k].y)), fmaxf(fabsf(v[k].z), fabsf(v[k].w))));
            const int e = prescale_exp(row_max(amax));
            const float inv = exp2i(-e);
            if (r == 0u) lds.scales[((tile & 1u) * KP + block) * PAIRS + i] = format_scale<SRC>() * exp2i(e);
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) {
                const float f[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
                union { uint2 u; _Float16 e[4]; } hi, lo;
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    const float t = f[n] * inv;
                    hi.e[n] = (_Float16)t;
                    lo.e[n] = (_Float16)split_rest(t, hi.e[n]);
                }
                // columns 64 k + 4 r .. + 3: eight of step s and lane quarter sq, their half r % 2
                const uint32_t c8 = 8u * k + r / 2u, s = fmt<SRC>() == F_IQ3_WORDS ? 4u * (c8 >> 4) + ((c8 >> 2) & 3u) : c8 & 7u, sq = fmt<SRC>() == F_IQ3_WORDS ? c8 & 3u : c8 >> 3;
                uint8_t *at = lds.x + ((SETS == 2 ? i / 16u : kPassTiles == 2u ? tile & 1u : 0u) * KP + block) * PANEL + (s * 64u + sq * 16u + (i & 15u)) * 16u + (r & 1u) * 8u;
                *reinterpret_cast<uint2 *>(at) = hi.u;
                *reinterpret_cast<uint2 *>(at + (SMALL ? 8u * 16u : 8192u)) = lo.u;      // (SMALL: the operand's rows 8 .. 15)
            }
        }
    };
    constexpr bool kAhead = NS <= (uint32_t)SETS;          // as far as the registers hold them
    Staged next;                                           // of tile `staged`
    uint32_t staged = tile0;                               // tiles below it are in LDS or were
    {
        Staged st;
        fetch_tile(st, first[0].p0, first[0].n);
        if constexpr (kAhead) fetch_tile(next, first[1].p0, first[1].n);
        __builtin_amdgcn_sched_barrier(0);
        if (tables) {
            if constexpr (small_tables<SRC>()) small_seeds.store(lds.entries, lds.signs, tid);
            else seeds.store(lds.entries, lds.signs, tid);
        }
        if (tid < n_info) lds.tiles[tid] = TileInfo{mat_of(info_e), info_p0, info_n};
        put_tile(st, staged++);
    }
    if constexpr (kPassTiles == 2u) {
        if (staged <= last_tile(p)) {
            if constexpr (!kAhead) fetch_tile(next, first[1].p0, first[1].n);
            put_tile(next, staged++);
        }
    }
    wave_lds_barrier();
    const LaneTables lt = lane_tables<SRC>(lds.entries, lds.signs, tid);
    const auto info_of = [&](uint32_t tile) { return uniform_info(lds.tiles[tile - tile0]); };
    const auto fetch_next = [&] { const TileInfo t = info_of(min(staged, tile0 + n_info - 1u)); fetch_tile(next, t.p0, t.n); };
    const auto advance = [&] {
        ahead.kb = 0u;
        ahead.p = following(ahead.p);
        ahead.before = ahead.info;
        ahead.info = info_of(ahead.p.tile + second(ahead.p));
    };
    const auto request = [&](Carried &c) {
        request_block(c, ahead.p, ahead.info.mat, ahead.kb);
        if (++ahead.kb == KP) advance();
    };
    if constexpr (KP <= 2u) advance();
    if constexpr (KP == 1u) request(c[1]);
    if constexpr (kAhead) { if (staged > tile0 + 1u) fetch_next(); }
    // Precision: as in gate/up, but a row's blocks are added up in f32, so the chains are half as long.
    constexpr uint32_t kChain = 2u;
    const float row_scale = SMALL && q >= 2u ? 4.8828125e-4f : 1.0f;      // of the lane's rows of the products
    float4_t sum[2][SETS];
    const auto clear = [&] {
#pragma unroll
        for (uint32_t m = 0; m < 2u; ++m)
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s) sum[m][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    };
    // adds the products of the block whose rows are in c
    const auto multiply = [&](const Carried &c, const uint8_t *x, const float *pair_scale) {
        const auto operand = [&](uint32_t s, uint32_t half, uint32_t step) { return *reinterpret_cast<const half8_t *>(x + s * KP * PANEL + half * 8192u + 1024u * step); };
        float4_t acc[2][SETS], low[2][SETS], block[2][SETS];
        float d[2];
        Entry e[2];
        half2_t f[2];
#pragma unroll
        for (uint32_t m = 0; m < 2u; ++m) {
            d[m] = quarter_d<SRC>(c.d[m]);
            if constexpr (SMALL) d[m] *= row_scale;
            e[m] = fetch_entry<SRC, 0u>(c.v[m], lt);
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s) acc[m][s] = low[m][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
        each_step([&](auto step) {
            constexpr uint32_t S = decltype(step)::value;
            // table reads run a step ahead of the products
            __builtin_amdgcn_sched_barrier(0);
            half8_t w[2], xh[SETS], xl[SETS];
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s) { xh[s] = operand(s, 0u, S); if constexpr (!SMALL) xl[s] = operand(s, 1u, S); }
#pragma unroll
            for (uint32_t m = 0; m < 2u; ++m) {
                if constexpr (steps_per_scale<SRC>() != 0u) { if constexpr (S % steps_per_scale<SRC>() == 0u) f[m] = step_scale<SRC, S>(c.v[m]); }
                w[m] = finish_entry<SRC>(e[m], f[m], lt);
                __builtin_amdgcn_sched_barrier(0);         // (the entry's registers take the next one)
                if constexpr (S < 7u) e[m] = fetch_entry<SRC, S + 1u>(c.v[m], lt);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (S && S % kChain == 0u) {
#pragma unroll
                for (uint32_t m = 0; m < 2u; ++m)
#pragma unroll
                    for (uint32_t s = 0; s < (uint32_t)SETS; ++s) {
                        block[m][s] = S == kChain ? acc[m][s] : block[m][s] + acc[m][s];
                        acc[m][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
                    }
            }
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s)
#pragma unroll
                for (uint32_t m = 0; m < 2u; ++m) acc[m][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh[s], w[m], acc[m][s], 0, 0, 0);
            if constexpr (!SMALL) {
#pragma unroll
                for (uint32_t s = 0; s < (uint32_t)SETS; ++s)
#pragma unroll
                    for (uint32_t m = 0; m < 2u; ++m) low[m][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl[s], w[m], low[m][s], 0, 0, 0);
            }
        });
#pragma unroll
        for (uint32_t s = 0; s < (uint32_t)SETS; ++s) {
            const float4_t ps = *reinterpret_cast<const float4_t *>(pair_scale + 16u * s + 4u * (SMALL ? q & 1u : q));
#pragma unroll
            for (uint32_t m = 0; m < 2u; ++m)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float both = SMALL ? block[m][s][t] + acc[m][s][t] : fmaf(low[m][s][t], 4.8828125e-4f, block[m][s][t] + acc[m][s][t]);
                    sum[m][s][t] = fmaf(both, d[m] * ps[t], sum[m][s][t]);
                }
        }
    };
    // No wave may skip a store (as in gate/up): of a wave without an item every one falls out of the range. A lane's distance from the first output of
    // the item is the same for every item. SMALL: the sums over high halves (lanes 0 .. 31) and over low ones meet, of the first row tile in the lower
    // lanes and of the second in the upper ones.
    const uint32_t out_at = 4u * ((SMALL ? 4u * (q & 1u) : 4u * q) * a.rows + (SMALL ? 16u * (q >> 1) : 0u) + r);
    const auto store_pass = [&] {
        const uint32_t item = p.j + wave - second(p) * ipt;
        const bool routed = uni(now.p0) < a.P;                 // (a tile is routed or shared as a whole)
        const auto buf = pair_rows(routed ? a.tmp : a.sh_tmp, routed ? now.p0 : now.p0 - a.P, wave < p.n ? now.n : 0u, a.rows);
        const uint32_t first_row = 4u * 32u * (wave < p.n ? item : 0u);
        if constexpr (SMALL) {
#pragma unroll
            for (uint32_t t = 0; t < 4u; ++t) {
                uint32_t x = __float_as_uint(sum[0][0][t]), y = __float_as_uint(sum[1][0][t] );
                swap32(x, y);
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(__uint_as_float(x) + __uint_as_float(y)), buf, out_at + 4u * t * a.rows, first_row, 0);
            }
        } else {
#pragma unroll
            for (uint32_t s = 0; s < (uint32_t)SETS; ++s)
#pragma unroll
                for (uint32_t t = 0; t < 4u; ++t)
#pragma unroll
                    for (uint32_t m = 0; m < 2u; ++m)
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sum[m][s][t]), buf, out_at + 4u * (16u * s + t) * a.rows, first_row + 64u * m, 0);
        }
    };
    const uint8_t *x_lane = lds.x + 16u * lane;
    uint32_t kb = 0u;
    clear();
    const auto block = [&](Carried &cc) {                  // false: the last one is done
        const uint32_t odd = (p.tile + second(p)) & 1u;
        if (wave < p.n) multiply(cc, x_lane + ((kPassTiles == 2u ? odd : 0u) * KP + kb) * PANEL, lds.scales + (odd * KP + kb) * PAIRS);
        request(cc);
        if (++kb < KP) return true;
        kb = 0u;
        store_pass();
        clear();
        if (last(p)) return false;
        p = following(p);
        now = KP == 1u ? info_of(p.tile + second(p)) : KP == 2u ? ahead.before : ahead.info;
        if (last_tile(p) >= staged) {
            wave_lds_barrier();                            // (nobody needs the tiles before the pass's any more)
            if constexpr (!kAhead) fetch_next();
            put_tile(next, staged++);
            if constexpr (kPassTiles == 2u) while (staged <= last_tile(p)) { fetch_next(); put_tile(next, staged++); }
            wave_lds_barrier();
            if constexpr (kAhead) fetch_next();
        }
        return true;
    };
    while (block(c[0]) && block(c[1])) {}
}

// SETS 1: the narrow tiles (list 2) of a chunk, SETS 2: the wide ones (list 1). Persistent workgroups, each with an equal run of the work.
// A launch that finds few wide tiles leaves them: the narrow one then takes every pair in tiles of 16 (list 0). Two launches where one would
// do cost 10 to 20 us (tables, the first tiles' activations, compute units without work at both ends); a wide tile saves a second decoding
// of its rows, which goes with their weights. So the line is a number of weights in wide tiles: 290 million for gate/up, 200 million for
// down, fitted while a tile of up to eight pairs cost as much as one of sixteen. Whole chunks since, us, by the line / never wide / wide wherever there are any:
//   gate/up  2048 x 768, 128 experts, eight a token: IQ2_XXS 300 tokens 160 / 149 / 160, 400 164 / 167 / 162, 700 246 / 252 / 245; F2 300 208 / 208 / 218, 512 297 / 292 / 298
//            1024 x 512, 200 experts, eight a token: IQ2_XXS 500 tokens 106 / 106 / 115, F2 700 151 / 152 / 162, IQ1_M 1000 183 / 182 / 194
//            2048 x 512, 512 experts, ten a token, Zipf: IQ2_XXS 512 tokens 232 / 236 / 233, 800 284 / 290 / 281; F2 512 266 / 264 / 272; own router, F2 1024 405 / 412 / 410
//   down     the same: 300 F2 208 / 206 / 214; 500 106 / 106 / 112, 700 F2 151 / 152 / 157; Zipf 512 F2 266 / 268 / 273, 1024 F2 405 / 413 / 408
// (runs of one side differ by 1 to 2 %). It lies right but for chunks whose wide tiles hold few pairs beyond sixteen (the first: 19 an expert), where a full tile
// and a small one are quicker: 7 % there. Wide down tiles of three blocks, and of four IQ3_S ones, fit the LDS beside small tables only; even so 2048 x 768, 128 experts, eight a token, raw
// rows take at 2048 tokens 239 us instead of 339 (IQ3_S), 196 / 242 (IQ2_XS), 181 / 191 (IQ1_M), whole calls of the pool 507 / 616, 543 / 595, 471 / 492
// and 467 / 491 (IQ2_XXS). The other formats' four blocks do not fit, and packed rows gain nothing.
template <int SRC, bool DOWN, uint32_t KP> constexpr bool has_wide() { return !DOWN || KP <= 2u || (layout<SRC>() == L_RAW && (KP == 3u || fmt<SRC>() == F_IQ3)); }
template <int SRC, int SETS, uint32_t KP> constexpr int down_src() { return SETS == 2 && KP > 2u ? SRC | SMALL_TABLES : SRC; }
template <int SRC, bool DOWN, uint32_t KP> uint32_t few_wide(uint32_t rows, uint32_t K) {
    return !has_wide<SRC, DOWN, KP>() ? ~0u : (DOWN ? 200000000u : 145000000u) / (rows * K) + 1u;
}
template <int SRC, bool DOWN, int SETS, uint32_t KP, bool SHORT>
__global__ __launch_bounds__((DOWN ? 64u * down_waves(SETS) : kGateUpThreads)) void staged_tiles_kernel(StagedArgs a) {
    __shared__ __attribute__((aligned(16))) std::conditional_t<DOWN, DownLds<down_src<SRC, SETS, KP>(), SETS, KP>, GateUpLds<SRC, SETS, KP>> lds;
    static_assert(sizeof(lds) <= 160u * 1024u, "what a compute unit has");
    const uint32_t n0 = a.n_tiles[0], n1 = a.n_tiles[1], n2 = a.n_tiles[2], b0 = a.n_tiles[3], b2 = a.n_tiles[4];      // (one trip)
    const bool few = n1 < a.few;
    if (SETS == 2 && few) return;
    const uint32_t l = SETS == 2 ? 1u : few ? 0u : 2u, off = l * a.list_stride;
    const uint32_t n_tiles = SETS == 2 ? n1 : few ? n0 : n2, n_big = SETS == 2 ? n_tiles : few ? b0 : b2;      // the others are small ones
    uint32_t per_tile = a.rows / (DOWN ? 32u : 16u * GateUp<SETS, DOWN ? 2u : KP>::NRT);
    if constexpr (DOWN && down_tiles_a_pass<SETS, KP>() == 1u) {
        // as many passes a tile as fill the rounds that the busiest workgroup has anyway
        const uint32_t least = (per_tile + down_waves(SETS) - 1u) / down_waves(SETS), rounds = (n_tiles * least + gridDim.x - 1u) / gridDim.x;
        per_tile = n_tiles ? min(per_tile / 4u, rounds * gridDim.x / n_tiles) : least;
    }
    const TileList list{a.tile_expert + off, a.tile_pair0 + off, a.tile_n + off};
    // workgroups are dealt round-robin over the eight XCDs: neighbouring runs (which share tiles) go to one XCD's L2
    const uint32_t G = gridDim.x, at = G % 8u == 0u ? (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u : blockIdx.x;
    // Equal shares of the time, small tiles and others on workgroups of their own: one that went from the others to the small ones began again with an empty
    // pipeline, 4 to 8 us behind all the rest (batch of 24 tokens, gate/up: ends at 41.6 us, the others at 34.4 on average). A unit of another tile takes 1.24
    // to 1.49 times as long as a small one's in gate/up and 1.07 to 1.29 times in down: gate/up, 2048 columns 2.10 and 1.61 us IQ2_XXS, 1.95 and 1.46 IQ1_M, 2.43 and
    // 1.96 IQ2_XS, 1024 columns 2.07 and 1.39; with popular experts, whose rows are at hand, 1.70 and 1.17; down 0.51 and 0.42, 0.49 and 0.38, 0.61 and 0.53, popular
    // 0.48 and 0.45. No one ratio fits all, so kCost is chosen among these by whole chunks: at 2048 columns 1.3, not 1.45 (F2, 512 tokens Zipf, two layers 521 and 547 us; the same
    // of IQ2_XXS, its pool chunk, 24 and 77 tokens within 2 %), at 1024 1.45 (150 tokens IQ1_M and 300 IQ2_XXS the same at 1.3); 512 columns as 1024, not measured. Parts
    // are too few for that: four to six a workgroup, one more of which lasts longer (150 tokens of 2048 x 768: 158 us undivided, 161 divided by whole rounds).
    const uint32_t w_big = n_big * per_tile, w_small = (n_tiles - n_big) * per_tile;
    uint32_t g_big = 0u;                                   // workgroups of the others; G: no such parting (no small tiles, or none but these)
    if (SETS == 2 || !w_small) g_big = G;
    else if constexpr (DOWN && down_tiles_a_pass<SETS, KP>() == 1u) g_big = G;
    else if (w_big) {
        constexpr float kCost = DOWN ? 1.15f : KP == 8u ? 1.3f : 1.45f;
        const float big = kCost * (float)w_big, small = (float)w_small;
        const uint32_t g = min(max((uint32_t)((float)G * big / (big + small)), 1u), G - 1u), more = min(g + 1u, G - 1u);
        const auto longest = [&](uint32_t n) { return fmaxf(big / (float)n, small / (float)(G - n)); };
        g_big = G == 1u ? G : longest(more) < longest(g) ? more : g;
    }
    const bool parted = g_big < G, mine_small = parted && at >= g_big;
    const uint32_t part_first = mine_small ? w_big : 0u, part = !parted ? w_big + w_small : mine_small ? w_small : w_big;
    const uint32_t part_at = mine_small ? at - g_big : at, part_groups = !parted ? G : mine_small ? G - g_big : g_big;
    const auto border = [&](uint32_t i) { return part_first + (uint32_t)((uint64_t)i * part / part_groups); };
    const uint32_t w0 = border(part_at), w1 = border(part_at + 1u);
    for (uint32_t from = w0; from < w1;) {                 // (a run of more than kTileInfos tiles in parts, small tiles apart)
        const bool small = from >= w_big;
        const uint32_t to = min(small ? w1 : min(w1, w_big), (from / per_tile + kTileInfos) * per_tile);
        if (from != w0) __syncthreads();
        if constexpr (DOWN) {
            constexpr int DSRC = down_src<SRC, SETS, KP>();
            if constexpr (SETS == 2) down_items<DSRC, SETS, KP, false>(a, list, per_tile, from, to, lds, from == w0);
            else if (small) down_items<DSRC, SETS, KP, true>(a, list, per_tile, from, to, lds, from == w0);
            else down_items<DSRC, SETS, KP, false>(a, list, per_tile, from, to, lds, from == w0);
        } else if constexpr (SETS == 1) {
            if (small) gateup_units<SRC, SETS, KP, SHORT, true>(a, list, from, to, lds, from == w0);
            else gateup_units<SRC, SETS, KP, SHORT, false>(a, list, from, to, lds, from == w0);
        } else gateup_units<SRC, SETS, KP, SHORT, false>(a, list, from, to, lds, from == w0);
        from = to;
    }
}

template <int SRC, bool DOWN, int SETS, uint32_t KP, bool SHORT = false>
hipError_t launch_staged_list(const StagedArgs &a, uint32_t grid, hipStream_t s) {
    REDHIP_LAUNCH((staged_tiles_kernel<SRC, DOWN, SETS, KP, SHORT>), dim3(grid), dim3(DOWN ? 64u * down_waves(SETS) : kGateUpThreads), 0, s, a);
    return hipGetLastError();
}
// wide: wide tiles that the chunk is expected to have; batch: it has so few tokens that still fewer would be slices
template <int SRC, bool DOWN, uint32_t KP>
hipError_t launch_staged_lists(StagedArgs a, uint32_t grid, uint32_t wide, bool batch, hipStream_t s) {
    a.few = few_wide<SRC, DOWN, KP>(a.rows, 256u * KP);
    hipError_t e = hipSuccess;
    if (wide < a.few) a.few = ~0u;                         // (without a wide launch the narrow one takes everything)
    if constexpr (has_wide<SRC, DOWN, KP>()) {
        if (a.few != ~0u) e = launch_staged_list<SRC, DOWN, 2, KP>(a, grid, s);
    }
    if constexpr (!DOWN && layout<SRC>() == L_TILED && KP >= 4u)
        if (batch) return e == hipSuccess ? launch_staged_list<SRC, DOWN, 1, KP, true>(a, grid, s) : e;
    return e == hipSuccess ? launch_staged_list<SRC, DOWN, 1, KP>(a, grid, s) : e;
}
template <int SRC>
hipError_t staged_gateup(const StagedArgs &a, uint32_t hidden, uint32_t grid, uint32_t wide, bool batch, hipStream_t s) {
    return hidden == 512u    ? launch_staged_lists<SRC, false, 2>(a, grid, wide, batch, s)
           : hidden == 1024u ? launch_staged_lists<SRC, false, 4>(a, grid, wide, batch, s)
                             : launch_staged_lists<SRC, false, 8>(a, grid, wide, batch, s);
}
template <int SRC>
hipError_t staged_down(const StagedArgs &a, uint32_t ffn, uint32_t grid, uint32_t wide, hipStream_t s) {
    if (ffn == 256u) return launch_staged_lists<SRC, true, 1>(a, grid, wide, false, s);
    if (ffn == 512u) return launch_staged_lists<SRC, true, 2>(a, grid, wide, false, s);
    if constexpr (layout<SRC>() == L_TILED) return hipErrorInvalidValue;      // (tile-major copies are made for ffn <= 512)
    else return ffn == 768u ? launch_staged_lists<SRC, true, 3>(a, grid, wide, false, s) : launch_staged_lists<SRC, true, 4>(a, grid, wide, false, s);
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
        case S_XXS: return staged_gateup<S_XXS>(a, hidden, grid, wide, c.batch, s);
        case S_XS: return staged_gateup<S_XS>(a, hidden, grid, wide, c.batch, s);
        case S_M: return staged_gateup<S_M>(a, hidden, grid, wide, c.batch, s);
        case S_ROWS_XXS: return staged_gateup<S_ROWS_XXS>(a, hidden, grid, wide, c.batch, s);
        case S_TILED_XXS: return staged_gateup<S_TILED_XXS>(a, hidden, grid, wide, c.batch, s);
        case S_TILED_XS: return staged_gateup<S_TILED_XS>(a, hidden, grid, wide, c.batch, s);
        case S_TILED_M: return staged_gateup<S_TILED_M>(a, hidden, grid, wide, c.batch, s);
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
