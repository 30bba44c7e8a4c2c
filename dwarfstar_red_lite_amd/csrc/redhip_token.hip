// One token's experts on raw GGUF rows (IQ2_XXS, IQ2_XS, IQ1_M, IQ3_S), read in place: gate and up rows with SwiGLU, then the down rows with
// the weighted sum over the experts (and the tail of a layer).
// Reference behaviour: native/redmetal_topk.m:1338-1415, :1858-1943 and native/redlite_native_reference.c:251-382.
//
// Both kernels are bound by latency: a token's rows are 9 MB, 2 us of memory, and the launches need what they read one round trip behind
// another (the slot's address, the rows, the codebook). So all requests of a wave are issued before the first is waited for, the tables are
// built while the rows are on their way, and no wave has more than one or two units: 16 rows times a block of 256 columns. The products run on v_mfma_f32_16x16x32_f16 with the
// weights as one operand, a quarter block of its row per lane (redhip_quarter.h); three of the 16 columns of the other operand hold the
// activation as fp16 terms x = t0 + t1 2^-11 + t2 2^-22, which is every bit of the f32 value, at no cost - one token leaves these
// columns empty. (Every bit down to 2^-26 of the block's largest value; below that the terms run out of exponents.)
// A token through ten IQ2_XS experts of 2048 x 512: gate/up 12.9 -> 9.1 us, down + sum 8.0 + 3.7 -> 6.4 us against one row per wave
// with scalar products, 32 columns per lane (the arithmetic on 2-byte-aligned pieces, and a grid entry looked up in memory behind the weights, took most of it).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "redhip_quarter.h"

namespace redhip {

namespace {

// the largest value of a wave, the same in every lane: rotations within sixteen lanes, then one value of each row of sixteen
__device__ __forceinline__ float wave_max(float v) {
    const auto dpp = [](float x, auto ctrl) { return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), decltype(ctrl)::value, 0xf, 0xf, false)); };
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0xB1>{}));         // quad_perm 1,0,3,2
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0x4E>{}));         // quad_perm 2,3,0,1
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0x124>{}));        // row_ror:4
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0x128>{}));        // row_ror:8
    const auto of = [&](int lane) { return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane)); };
    return fmaxf(fmaxf(of(0), of(16)), fmaxf(of(32), of(48)));
}

// lane's four consecutive activations of a block -> three planes of 256 fp16 terms in LDS; returns the block's power of two
__device__ __forceinline__ float store_terms(float4 x, _Float16 *planes, uint32_t lane) {
    float amax = fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)));
    const int e = prescale_exp(wave_max(amax));
    const float inv = exp2i(-e), v[4] = {x.x, x.y, x.z, x.w};
    union { uint2 u; _Float16 h[4]; } t[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float rest = v[i] * inv;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            t[k].h[i] = (_Float16)rest;
            rest = split_rest(rest, t[k].h[i]);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<uint2 *>(planes + k * 256 + 4 * lane) = t[k].u;
    return exp2i(e);
}

// eight activation terms of step s for operand row i = lane % 16 (rows beyond the third repeat it: their products are not used)
__device__ __forceinline__ half8_t term_operand(const _Float16 *planes, uint32_t s, uint32_t i, uint32_t q) {
    return *reinterpret_cast<const half8_t *>(planes + min(i, 2u) * 256u + 64u * q + 8u * s);
}

// one unit: 16 rows (row r of lanes r, r + 16, ..) times a block; the sum of row r in lanes 0 .. 15
template <int SRC>
__device__ __forceinline__ float unit_product(const Quarter &v, uint2 d, const _Float16 *planes, uint32_t i, uint32_t q, const LaneTables &lt) {
    float4_t acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};      // (half of the block each: half as many roundings behind one another)
    half2_t f{};
    each_step([&](auto step) {
        constexpr uint32_t s = decltype(step)::value;
        if constexpr (s % steps_per_scale<SRC>() == 0u) f = step_scale<SRC, s>(v);
        acc[s >> 2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(term_operand(planes, s, i, q), finish_entry<SRC>(fetch_entry<SRC, s>(v, lt), f, lt), acc[s >> 2], 0, 0, 0);
    });
    acc[0] += acc[1];
    return (acc[0][0] + (acc[0][1] + acc[0][2] * 4.8828125e-4f) * 4.8828125e-4f) * quarter_d<SRC>(d);
}

// act[slot][r] = SiLU(gate[r] . x) * (up[r] . x). Sixteen waves: KP of them, one block of 256 columns each (or every KP-th), share 16 gate
// rows, as many the up rows; eight blocks or more take KP = 8, fewer KP = 4 and two groups of rows per workgroup.
template <int SRC, uint32_t KP>
__global__ __launch_bounds__(1024) void token_gateup_kernel(const uint64_t *table, const uint8_t *base, const float *x, const float *x1, float *act, uint32_t x_split,
                                                            uint32_t n_block, uint32_t ffn, uint64_t up_delta, const int8_t *grid) {
    constexpr uint32_t G = 8u / KP;
    __shared__ __attribute__((aligned(16))) uint8_t entries[small_entry_bytes<SRC>()];
    __shared__ __attribute__((aligned(16))) uint32_t signs[sign_bytes<SRC>() / 4u + 4u];
    __shared__ __attribute__((aligned(16))) _Float16 planes[16][768];
    __shared__ float part[16][16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4, slot = blockIdx.y;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), k0 = wave % KP, up = (wave / KP) & 1u, group = wave / (2u * KP);
    SmallSeeds<SRC, 1024u> seeds;
    seeds.request(tid, grid);
    const float *xin = x1 && slot >= x_split ? x1 : x;
    const uint32_t kf = k0 < n_block ? k0 : n_block - 1u;              // (a wave without a block requests the last and uses nothing of it)
    float4 xv = reinterpret_cast<const float4 *>(xin)[64u * kf + lane];
    const uint8_t *gate = table ? reinterpret_cast<const uint8_t *>(table[slot]) : base;
    const uint8_t *row = gate + (up ? up_delta : 0u) + (uint64_t)((blockIdx.x * G + group) * 16u + r) * (n_block * src_block<SRC>());
    Quarter v;
    uint2 d;
    load_quarter<SRC, 1u>(row, nullptr, nullptr, 0u, kf, q, v, d);
    seeds.store(entries, signs, tid);
    float scale = store_terms(xv, planes[wave], lane);
    __syncthreads();
    const LaneTables lt = lane_tables<SRC>(entries, signs, tid);
    float sum = 0.0f;
    for (uint32_t k = k0; k < n_block;) {
        sum += unit_product<SRC>(v, d, planes[wave], r, q, lt) * (scale * format_scale<SRC>());
        k += KP;
        if (k >= n_block) break;
        load_quarter<SRC, 1u>(row, nullptr, nullptr, 0u, k, q, v, d);
        xv = reinterpret_cast<const float4 *>(xin)[64u * k + lane];
        scale = store_terms(xv, planes[wave], lane);
    }
    if (lane < 16u) part[wave][r] = sum;
    __syncthreads();
    if (tid < G * 16u) {
        const float(*p)[16] = part + (tid >> 4) * 2u * KP;
        float g = p[0][r], u = p[KP][r];
#pragma unroll
        for (uint32_t k = 1; k < KP; ++k) { g += p[k][r]; u += p[KP + k][r]; }
        act[(uint64_t)slot * ffn + (blockIdx.x * G + (tid >> 4)) * 16u + r] = (g / (1.0f + expf(-g))) * u;
    }
}

// out[i] = sum_k weights[k] * (down_k[row_start + i] . act_k) (weights == nullptr: one expert, weight 1).
// With a tail, out[i] and layer_out[i] = resid[i] + (the sum + shared[i] * scalar[0]).
// T / 64 waves: uw of them share 16 rows, unit (expert, block) number w, w + uw, .. each; the units' sums meet in LDS.
struct TokenDownArgs {
    const uint64_t *table;
    const uint8_t *base;                 // down matrix of an expert at base or table[k], plus down_off
    const float *act, *weights;
    float *out;
    uint64_t down_off;
    uint32_t n_block, block_magic, units, uw, row_start, row_end;      // (u * block_magic) >> 16 = u / n_block
    const float *resid, *shared, *scalar;
    float *layer_out;
    const int8_t *grid;
};
constexpr uint32_t kTokenUnits = 256u, kTokenExperts = 64u;
template <int SRC, uint32_t T>
__global__ __launch_bounds__(T) void token_down_kernel(TokenDownArgs a) {
    constexpr uint32_t W = T / 64u;
    __shared__ __attribute__((aligned(16))) uint8_t entries[small_entry_bytes<SRC>()];
    __shared__ __attribute__((aligned(16))) uint32_t signs[sign_bytes<SRC>() / 4u + 4u];
    __shared__ __attribute__((aligned(16))) _Float16 planes[W][768];
    __shared__ float part[T == 1024u ? kTokenUnits : W * 8u][16];      // (T 256: at most eight units, W groups of rows)
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, q = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = wave / a.uw, u0 = wave % a.uw, groups = W / a.uw;
    const uint32_t row0 = a.row_start + (blockIdx.x * groups + group) * 16u, row = min(row0 + r, a.row_end - 1u);      // (surplus rows repeat the last; not stored)
    SmallSeeds<SRC, T> seeds;
    seeds.request(tid, a.grid);
    const uint64_t row_off = a.down_off + (uint64_t)row * (a.n_block * src_block<SRC>());
    Quarter v;
    uint2 d;
    float4 xv;
    float w;
    const auto request = [&](uint32_t u) {
        const uint32_t e = (u * a.block_magic) >> 16, k = u - e * a.n_block;
        xv = reinterpret_cast<const float4 *>(a.act)[64u * u + lane];
        w = a.weights ? a.weights[e] : 1.0f;
        load_quarter<SRC, 1u>((a.table ? reinterpret_cast<const uint8_t *>(a.table[e]) : a.base) + row_off, nullptr, nullptr, 0u, k, q, v, d);
    };
    request(u0 < a.units ? u0 : a.units - 1u);
    seeds.store(entries, signs, tid);
    float scale = store_terms(xv, planes[wave], lane) * format_scale<SRC>() * w;
    __syncthreads();
    const LaneTables lt = lane_tables<SRC>(entries, signs, tid);
    for (uint32_t u = u0; u < a.units;) {
        const Quarter cv = v;
        const uint2 cd = d;
        const uint32_t next = u + a.uw;
        if (next < a.units) request(next);
        const float s = unit_product<SRC>(cv, cd, planes[wave], r, q, lt) * scale;
        if (lane < 16u) part[group * a.units + u][r] = s;
        if (next < a.units) scale = store_terms(xv, planes[wave], lane) * format_scale<SRC>() * w;
        u = next;
    }
    __syncthreads();
    if (wave < groups) {                                               // every fourth unit per lane, then the four sums
        float sum = 0.0f;
        for (uint32_t u = q; u < a.units; u += 4u) sum += part[wave * a.units + u][r];
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        const uint32_t at = a.row_start + (blockIdx.x * groups + wave) * 16u + r;
        if (lane < 16u && at < a.row_end) {
            const uint32_t i = at - a.row_start;
            if (a.layer_out) {
                sum = a.resid[i] + (sum + a.shared[i] * a.scalar[0]);
                a.layer_out[i] = sum;
            }
            a.out[i] = sum;
        }
    }
}

int token_src(uint32_t type) { return type == T_IQ2_XXS ? F_XXS : type == T_IQ2_XS ? F_XS : type == T_IQ1_M ? F_M : type == T_IQ3_S ? F_IQ3 : -1; }

template <int F>
hipError_t token_gateup(const ExpertSet &ex, uint32_t n_slot, uint32_t hidden, uint32_t ffn, const float *x, const float *x1, uint32_t x_split, float *act, hipStream_t s) {
    constexpr int SRC = F | SMALL_TABLES;
    const uint32_t nb = hidden / 256u;
    const int8_t *grid = caller_grid_device(ex.gate_up_type);
    if (nb > 4u) REDHIP_LAUNCH((token_gateup_kernel<SRC, 8u>), dim3(ffn / 16u, n_slot), dim3(1024), 0, s, ex.table, ex.base, x, x1, act, x_split, nb, ffn, ex.gate_bytes, grid);
    else REDHIP_LAUNCH((token_gateup_kernel<SRC, 4u>), dim3(ffn / 32u, n_slot), dim3(1024), 0, s, ex.table, ex.base, x, x1, act, x_split, nb, ffn, ex.gate_bytes, grid);
    return hipGetLastError();
}
template <int F>
hipError_t token_down(TokenDownArgs a, hipStream_t s) {
    constexpr int SRC = F | SMALL_TABLES;
    const uint32_t rows = a.row_end - a.row_start;
    if (a.units <= 8u) {                                               // few units (one expert): smaller workgroups, more of them
        a.uw = a.units <= 1u ? 1u : a.units <= 2u ? 2u : 4u;
        const uint32_t per = 16u * (4u / a.uw);
        REDHIP_LAUNCH((token_down_kernel<SRC, 256u>), dim3((rows + per - 1u) / per), dim3(256), 0, s, a);
    } else {
        a.uw = 16u;
        REDHIP_LAUNCH((token_down_kernel<SRC, 1024u>), dim3((rows + 15u) / 16u), dim3(1024), 0, s, a);
    }
    return hipGetLastError();
}

}  // namespace

// x is read as float4; the units of a down row and the experts' weights have to fit the kernel's LDS
bool token_rows_supported(uint32_t gate_up_type, uint32_t down_type, uint32_t top_k, uint32_t hidden, uint32_t ffn, const float *x, const float *x1) {
    return token_src(gate_up_type) >= 0 && token_src(down_type) >= 0 && top_k && top_k <= kTokenExperts && hidden && hidden % 256u == 0u && ffn && ffn % 256u == 0u &&
           (uint64_t)top_k * (ffn / 256u) <= kTokenUnits && !((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(x1)) & 15u);
}

hipError_t launch_token_gateup(const ExpertSet &ex, uint32_t n_slot, uint32_t hidden, uint32_t ffn, const float *x, const float *x1, uint32_t x_split, float *act, hipStream_t s) {
    switch (token_src(ex.gate_up_type)) {
        case F_XXS: return token_gateup<F_XXS>(ex, n_slot, hidden, ffn, x, x1, x_split, act, s);
        case F_XS: return token_gateup<F_XS>(ex, n_slot, hidden, ffn, x, x1, x_split, act, s);
        case F_M: return token_gateup<F_M>(ex, n_slot, hidden, ffn, x, x1, x_split, act, s);
        case F_IQ3: return token_gateup<F_IQ3>(ex, n_slot, hidden, ffn, x, x1, x_split, act, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_token_down(const ExpertSet &ex, const float *weights, uint32_t top_k, uint32_t ffn, uint32_t row_start, uint32_t row_count, const float *act, float *out,
                             const TokenTail *tail, hipStream_t s) {
    TokenDownArgs a{};
    a.table = ex.table; a.base = ex.base; a.act = act; a.weights = weights;
    a.out = tail ? tail->x : out;
    a.down_off = ex.gate_bytes + ex.up_bytes;
    a.n_block = ffn / 256u; a.units = top_k * a.n_block;
    a.block_magic = (65536u + a.n_block - 1u) / a.n_block;             // (exact below kTokenUnits)
    a.row_start = row_start; a.row_end = row_start + row_count;
    if (tail) { a.resid = tail->resid; a.shared = tail->shared; a.scalar = tail->scalar; a.layer_out = tail->layer_out; }
    a.grid = caller_grid_device(ex.down_type);
    switch (token_src(ex.down_type)) {
        case F_XXS: return token_down<F_XXS>(a, s);
        case F_XS: return token_down<F_XS>(a, s);
        case F_M: return token_down<F_M>(a, s);
        case F_IQ3: return token_down<F_IQ3>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace redhip
