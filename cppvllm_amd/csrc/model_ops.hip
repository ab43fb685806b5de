// gfx950 kernels for the model ops around the attention path: SwiGLU, the token sampler
// (greedy arg-max and Gumbel-max), token feedback and the embedding gather.
//
// These feed or consume the hot path once per layer (SwiGLU) or once per step (the rest); they
// are HBM/launch bound, so each is one coalesced pass with 16-byte accesses.
//
// Numerics (matched bit for bit by the CPU oracle):
//   swiglu : silu = round_T( (float)( g / (1 + exp(-g)) ) evaluated in double ),
//            out = round_T( silu * u ) in float — the reference's rounding points
//            (kernels/fused_ops.cu:210-219) with the exponential evaluated in double so that the
//            result does not depend on the exp implementation's last float ulp.
//   sampler: arg-max with the lowest index winning ties (kernels/fused_ops.cu:302-303); the
//            Gumbel score of a sampling row is (float)(x*inv_t - log(max(-log(u), 1e-10))) in
//            double, u from Philox-4x32-10 (Salmon et al., SC'11) with the counter layout of
//            kernels/fused_ops.cu:327-330 (index/4, row, offset).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "cvh_device.h"

namespace cvh {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 ld_nt(const void* p) { return __builtin_nontemporal_load(static_cast<const u32x4*>(p)); }

// ---- SwiGLU ---------------------------------------------------------------------------------

// The bf16 SiLU table in LDS: the gates with 2^-15 <= |g| < 2^7, both signs, 11 KB of the 128 KB table
// (a gate outside, which is rare, reads the whole table in global memory).
constexpr int kLutFirst = (127 - 15) << 7, kLutGates = 22 << 7;
__device__ __forceinline__ void load_silu_lut(uint16_t* lut) {
    constexpr int kPieces = kLutGates / 8;       // 16-byte pieces per sign
    for (int i = threadIdx.x; i < 2 * kPieces; i += blockDim.x) {
        const int neg = i >= kPieces;
        reinterpret_cast<uint4*>(lut)[i] =
                *reinterpret_cast<const uint4*>(kSiluBf16 + (neg ? 0x8000 : 0) + kLutFirst + (i - (neg ? kPieces : 0)) * 8);
    }
}
// out word: silu(gate) * up of the two bf16 in g and u
__device__ __forceinline__ uint32_t silu_mul_bf16x2(const uint16_t* lut, uint32_t g, uint32_t u) {
    const uint32_t a = g & 0x7fffu, b = (g >> 16) & 0x7fffu;
    const uint32_t ia = a - kLutFirst, ib = b - kLutFirst;
    uint32_t sa = lut[min(ia, kLutGates - 1u) + ((g & 0x8000u) ? kLutGates : 0)];
    uint32_t sb = lut[min(ib, kLutGates - 1u) + ((g & 0x80000000u) ? kLutGates : 0)];
    if (max(ia, ib) >= kLutGates) {
        if (ia >= kLutGates) sa = kSiluBf16[g & 0xffffu];
        if (ib >= kLutGates) sb = kSiluBf16[g >> 16];
    }
    return pack_bf16x2(bf16_bits_to_f32(sa) * bf16_bits_to_f32(u & 0xffffu),
                       bf16_bits_to_f32(sb) * __uint_as_float(u & 0xffff0000u));
}

// bf16, I % 8 == 0, more than kSwigluDirect 8-output pieces: 8 consecutive outputs of a row per thread and
// turn (two 16-byte loads, one 16-byte store), the SiLU looked up in LDS. With the lookups in the global
// table the kernel was bound by their gathers (64 lines per load): 4096 x 3072 outputs 21.4 us, 13.2 us now
// (75 MB, 5.7 TB/s). Workgroups of 1024 threads walk the outputs, at most two per CU, so that the table is
// loaded at most 512 times. With fewer pieces the table's load is not earned back: 64 x 3072 outputs 2.6 us by
// swiglu_kernel, 3.3 this way; 680 x 1536 (130560 pieces) 3.3 and 3.6. Above, it is: 512 x 3072 (196608) 3.8 us, 4.2
// when the bf16 kernel was the direct one.
constexpr int kSwigluThreads = 1024, kSwigluBlocks = 512, kSwigluDirect = 1 << 17;
__global__ __launch_bounds__(kSwigluThreads) void swiglu_bf16_kernel(uint16_t* __restrict__ out,
                                                                     const uint16_t* __restrict__ gu, int64_t n8, int I) {
    __shared__ __align__(16) uint16_t lut[2 * kLutGates];
    const uint32_t per_row = static_cast<uint32_t>(I) >> 3;
    const int64_t step = static_cast<int64_t>(gridDim.x) * kSwigluThreads;
    int64_t k = static_cast<int64_t>(blockIdx.x) * kSwigluThreads + threadIdx.x;
    u32x4 g = {0, 0, 0, 0}, u = g;
    auto place = [&](int64_t at, int64_t& r, uint32_t& c) {
        if (n8 <= 0xffffffffll) {                 // one 32-bit division instead of a 64-bit one
            r = static_cast<uint32_t>(at) / per_row;
            c = static_cast<uint32_t>(at) - static_cast<uint32_t>(r) * per_row;
        } else {
            r = at / per_row;
            c = static_cast<uint32_t>(at - r * per_row);
        }
    };
    auto load = [&](int64_t at) {
        int64_t r;
        uint32_t c;
        place(at, r, c);
        const uint16_t* p = gu + r * 2 * I + c * 8;
        g = ld_nt(p);
        u = ld_nt(p + I);
    };
    if (k < n8) load(k);
    load_silu_lut(lut);
    __syncthreads();
    for (; k < n8; k += step) {
        const u32x4 gk = g, uk = u;
        if (k + step < n8) load(k + step);
        uint4 o;
        o.x = silu_mul_bf16x2(lut, gk.x, uk.x);
        o.y = silu_mul_bf16x2(lut, gk.y, uk.y);
        o.z = silu_mul_bf16x2(lut, gk.z, uk.z);
        o.w = silu_mul_bf16x2(lut, gk.w, uk.w);
        *reinterpret_cast<uint4*>(out + k * 8) = o;
    }
}

// I % 8 == 0, f16, f32 and few bf16 outputs: one thread per 8 consecutive outputs of a row.
template <int DT>
__global__ __launch_bounds__(256) void swiglu_kernel(typename Elem<DT>::T* __restrict__ out,
                                                     const typename Elem<DT>::T* __restrict__ gu, int64_t n8, int I) {
    using T = typename Elem<DT>::T;
    const int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n8) return;
    const int per_row = I >> 3;
    const int64_t r = k / per_row;
    const int c = static_cast<int>(k - r * per_row) << 3;
    const T* g = gu + r * 2 * I + c;
    const T* u = g + I;
    T* o = out + r * I + c;
    T gv[8], uv[8], ov[8];
    constexpr int kWords = 8 * sizeof(T) / 16;
#pragma unroll
    for (int j = 0; j < kWords; ++j) {
        reinterpret_cast<u32x4*>(gv)[j] = ld_nt(reinterpret_cast<const u32x4*>(g) + j);
        reinterpret_cast<u32x4*>(uv)[j] = ld_nt(reinterpret_cast<const u32x4*>(u) + j);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ov[j] = Elem<DT>::store(silu_mul<DT>(Elem<DT>::load(gv[j]), Elem<DT>::load(uv[j])));
#pragma unroll
    for (int j = 0; j < kWords; ++j) reinterpret_cast<u32x4*>(o)[j] = reinterpret_cast<const u32x4*>(ov)[j];
}

// Any I: one thread per output.
template <int DT>
__global__ __launch_bounds__(256) void swiglu_scalar_kernel(typename Elem<DT>::T* __restrict__ out,
                                                            const typename Elem<DT>::T* __restrict__ gu, int64_t n,
                                                            int I) {
    const int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int64_t r = k / I;
    const int i = static_cast<int>(k - r * I);
    out[k] = Elem<DT>::store(silu_mul<DT>(Elem<DT>::load(gu[r * 2 * I + i]), Elem<DT>::load(gu[r * 2 * I + I + i])));
}

// ---- Sampler ----------------------------------------------------------------------------------
// Design: every candidate becomes one 64-bit key whose unsigned order is the selection order,
//   key = order32(score) << 32 | (0xFFFFFFFF - index),
// so "largest score, lowest index on ties" is a plain unsigned max and a row's winner is the max
// over all its keys. order32 maps float bit patterns to an unsigned order (negatives bit-flipped,
// positives with the sign bit set) and sends NaN below every number, so a NaN never wins. The
// search starts from the key of (-inf, index 0x7FFFFFFF): an all -inf row then gives index 0 and
// an all-NaN row 0x7FFFFFFF, as the reference's (value, index) scan does (kernels/fused_ops.cu:
// 300-306).
// Work split: a row, or its part when few rows would leave CUs idle (sample_parts), is one workgroup
// of kSampleWaves waves; wave w owns a contiguous slice of S logits (S a multiple of 8), and its lanes
// read 8 logits (16 bytes of bf16) at a time, lane-consecutive, so one load instruction of a wave
// covers 1 KB contiguous. Each lane folds its keys with a 64-bit max; the wave folds them with a
// DPP/permlane butterfly on the two 32-bit halves; wave leaders fold into one LDS word with
// ds_max_u64. Greedy rows are bound by the latency of a few loads per wave, sampling rows by the
// integer multiplies of Philox (20 per 4 candidates, a quarter of the VALU rate).
constexpr int kSampleWaves = 16;

// Philox-4x32 with 10 rounds (Random123's philox4x32_10): multipliers 0xD2511F53 / 0xCD9E8D57,
// Weyl key increments 0x9E3779B9 / 0xBB67AE85.
__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        const uint32_t hi0 = __umulhi(0xD2511F53u, c[0]), lo0 = 0xD2511F53u * c[0];
        const uint32_t hi1 = __umulhi(0xCD9E8D57u, c[2]), lo1 = 0xCD9E8D57u * c[2];
        const uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = lo1;
        c[2] = n2;
        c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

__device__ __forceinline__ uint64_t rank_key(float s, uint32_t index) {
    uint32_t b = __float_as_uint(s);
    if (b == 0x80000000u) b = 0u;                  // -0.0 ties with +0.0 (lower index wins)
    uint32_t o = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    if ((b & 0x7fffffffu) > 0x7f800000u) o = 0u;   // NaN: below -inf
    return (static_cast<uint64_t>(o) << 32) | (0xFFFFFFFFu - index);
}
__device__ __forceinline__ uint32_t key_index(uint64_t k) { return 0xFFFFFFFFu - static_cast<uint32_t>(k); }
__device__ __forceinline__ uint64_t kmax(uint64_t a, uint64_t b) { return a > b ? a : b; }

// Gumbel perturbation of logit x with the 32-bit uniform word r: u = ((r >> 8) + 0.5) / 2^24 (exact
// in float), score = x / t - log(max(-log u, 1e-10)) evaluated in double and rounded to float.
__device__ __forceinline__ float perturbed(float x, float inv_t, uint32_t r) {
    const float u = (static_cast<float>(r >> 8) + 0.5f) * (1.0f / 16777216.0f);
    const double g = -log(fmax(-log(static_cast<double>(u)), 1e-10));
    return static_cast<float>(static_cast<double>(x) * inv_t + g);
}

template <int CTRL> __device__ __forceinline__ uint64_t dpp64(uint64_t v) {
    const uint32_t lo = __builtin_amdgcn_mov_dpp(static_cast<int>(static_cast<uint32_t>(v)), CTRL, 0xF, 0xF, true);
    const uint32_t hi = __builtin_amdgcn_mov_dpp(static_cast<int>(static_cast<uint32_t>(v >> 32)), CTRL, 0xF, 0xF, true);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}
// Max over the 64 lanes (every lane active): quad DPP, then mirrors (exact once quads / halves are
// uniform), then the gfx950 permlane16/32 swaps across rows.
__device__ __forceinline__ uint64_t wave_kmax(uint64_t v) {
    v = kmax(v, dpp64<0xB1>(v));
    v = kmax(v, dpp64<0x4E>(v));
    v = kmax(v, dpp64<0x141>(v));
    v = kmax(v, dpp64<0x140>(v));
    uint32_t lo = static_cast<uint32_t>(v), hi = static_cast<uint32_t>(v >> 32);
    auto l16 = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    auto h16 = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    v = kmax((static_cast<uint64_t>(h16[0]) << 32) | l16[0], (static_cast<uint64_t>(h16[1]) << 32) | l16[1]);
    lo = static_cast<uint32_t>(v);
    hi = static_cast<uint32_t>(v >> 32);
    auto l32 = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    auto h32 = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return kmax((static_cast<uint64_t>(h32[0]) << 32) | l32[0], (static_cast<uint64_t>(h32[1]) << 32) | l32[1]);
}

// The 8 logits at [j, j+8) of a row as float; positions past V read as -inf (never selected:
// the caller does not fold them).
template <int LDT>
__device__ __forceinline__ void logits8(const char* row, int j, int V, float* x) {
    if (j + 8 <= V && (V & 7) == 0) {
        if constexpr (LDT == CVH_DTYPE_F32) {
            const u32x4 a = ld_nt(row + static_cast<size_t>(j) * 4);
            const u32x4 b = ld_nt(row + static_cast<size_t>(j) * 4 + 16);
            x[0] = __uint_as_float(a.x); x[1] = __uint_as_float(a.y); x[2] = __uint_as_float(a.z); x[3] = __uint_as_float(a.w);
            x[4] = __uint_as_float(b.x); x[5] = __uint_as_float(b.y); x[6] = __uint_as_float(b.z); x[7] = __uint_as_float(b.w);
        } else {
            const u32x4 a = ld_nt(row + static_cast<size_t>(j) * 2);
            const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[2 * e] = bf16_bits_to_f32(w[e] & 0xffffu);
                x[2 * e + 1] = bf16_bits_to_f32(w[e] >> 16);
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (j + e >= V) { x[e] = -INFINITY; continue; }
            if constexpr (LDT == CVH_DTYPE_F32) x[e] = reinterpret_cast<const float*>(row)[j + e];
            else x[e] = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(row)[j + e]);
        }
    }
}

// Greedy rows: the best key of logits [lo, hi) (this lane's share).
template <int LDT>
__device__ __forceinline__ uint64_t scan_greedy(const char* row, int lo, int hi, int V, int lane) {
    uint64_t best = rank_key(-INFINITY, 0x7fffffffu);
    for (int j = lo + 8 * lane; j < hi; j += 8 * 64) {
        float x[8];
        logits8<LDT>(row, j, V, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (j + e >= hi) break;
            best = kmax(best, rank_key(x[e], static_cast<uint32_t>(j + e)));
        }
    }
    return best;
}

// Sampling rows. A Gumbel score takes two double logarithms (~300 instructions), but only the row's
// winner has to be known exactly: a first pass scores every candidate in float (screen_score, within
// screen_tol of the double score), and the double scores are computed only where the float one comes
// within the tolerance of the largest, usually for one 8-logit chunk of one lane. The winner is the
// one that scoring everything in double gives. 48 rows of 151936 bf16 logits (half of them
// greedy): 227 us when every candidate was scored in double by one workgroup a row, 18.6 us now (five
// workgroups a row) plus two 2-4 us launches that clear and decode the rows' keys.
__device__ __forceinline__ float screen_score(float x, float inv_t, uint32_t r) {
    const float u = (static_cast<float>(r >> 8) + 0.5f) * (1.0f / 16777216.0f);   // as perturbed() has it
    // -log u: near 1 by its series in 1 - u (exact for u >= 1/2; remainder < 4e-6 relative below
    // 1/16), elsewhere by the hardware log2, whose absolute error is there small against the result
    const float w = 1.0f - u;
    const float near1 = w * __builtin_fmaf(w, __builtin_fmaf(w, __builtin_fmaf(w, 0.25f, 1.0f / 3.0f), 0.5f), 1.0f);
    const float e = w < 0.0625f ? near1 : -0.693147181f * __builtin_amdgcn_logf(u);
    return __builtin_fmaf(x, inv_t, -0.693147181f * __builtin_amdgcn_logf(fmaxf(e, 1e-10f)));
}
// Bound on |screen_score - perturbed|: under 1e-5 from the logarithms and 2^-23 of the score from the
// roundings to float, with a margin of ten and four.
__device__ __forceinline__ float screen_tol(float a) { return __builtin_fmaf(fabsf(a), 0x1p-21f, 1e-4f); }

// The uniform words of candidates j .. j + 7 (j % 8 == 0): Philox counter (index / 4, row, offset), one
// block per 4 indices.
__device__ __forceinline__ void words4(int j, int r, uint64_t seed, uint64_t offset, uint32_t (&c)[4]) {
    c[0] = static_cast<uint32_t>(j >> 2);
    c[1] = static_cast<uint32_t>(r);
    c[2] = static_cast<uint32_t>(offset);
    c[3] = static_cast<uint32_t>(offset >> 32);
    philox4x32_10(c, static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32));
}

// The best key of candidates [j, min(j + 8, hi)), scored in double.
template <int LDT>
__device__ __forceinline__ uint64_t exact_chunk(const char* row, int j, int hi, int r, float inv_t, uint64_t seed,
                                                uint64_t offset) {
    uint64_t best = rank_key(-INFINITY, 0x7fffffffu);
#pragma unroll 1
    for (int h = 0; h < 8; h += 4) {
        uint32_t c[4];
        words4(j + h, r, seed, offset, c);
#pragma unroll 1
        for (int e = 0; e < 4 && j + h + e < hi; ++e) {
            const int i = j + h + e;
            const uint32_t w = e == 0 ? c[0] : e == 1 ? c[1] : e == 2 ? c[2] : c[3];
            const float x = LDT == CVH_DTYPE_F32 ? reinterpret_cast<const float*>(row)[i]
                                                 : bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(row)[i]);
            best = kmax(best, rank_key(perturbed(x, inv_t, w), static_cast<uint32_t>(i)));
        }
    }
    return best;
}

// One workgroup's best key of a sampling row's candidates [lo, hi) per wave; wave_top: LDS, one float
// per wave. Every wave of the workgroup calls it.
template <int LDT>
__device__ __forceinline__ uint64_t scan_gumbel(const char* row, int lo, int hi, int V, int lane, int wave, int r,
                                                float inv_t, uint64_t seed, uint64_t offset, float* wave_top) {
    // this lane's largest screen score, the chunk that holds it, and the largest of its other chunks
    float top = -INFINITY, rest = -INFINITY;
    int top_j = lo;
    for (int j = lo + 8 * lane; j < hi; j += 8 * 64) {
        float x[8];
        logits8<LDT>(row, j, V, x);            // -inf past V
        float m = -INFINITY;
#pragma unroll
        for (int h = 0; h < 8; h += 4) {
            uint32_t c[4];
            words4(j + h, r, seed, offset, c);
#pragma unroll
            for (int e = 0; e < 4; ++e) m = fmaxf(m, screen_score(x[h + e], inv_t, c[e]));   // a NaN never counts
        }
        if (m > top) {
            rest = top;
            top = m;
            top_j = j;
        } else {
            rest = fmaxf(rest, m);
        }
    }
    const float wt = xor_max<64>(top);
    if (lane == 0) wave_top[wave] = wt;
    __syncthreads();
    float best_top = wave_top[lane & (kSampleWaves - 1)];
    best_top = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, xor_max<64>(best_top))));
    uint64_t k = rank_key(-INFINITY, 0x7fffffffu);
    if (fabsf(best_top) < 1e30f) {
        const float floor = best_top - screen_tol(best_top);
        if (rest + screen_tol(rest) >= floor) {                   // several chunks of the lane are in reach
            for (int j = lo + 8 * lane; j < hi; j += 8 * 64)
                k = kmax(k, exact_chunk<LDT>(row, j, hi, r, inv_t, seed, offset));
        } else if (top + screen_tol(top) >= floor) {
            k = exact_chunk<LDT>(row, top_j, hi, r, inv_t, seed, offset);
        }
    } else if (best_top == -INFINITY) {        // no candidate above -inf: the first that is no NaN wins
        for (int j = lo + 8 * lane; j < hi; j += 8 * 64) {
            float x[8];
            logits8<LDT>(row, j, V, x);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (j + e < hi && x[e] * inv_t == -INFINITY) k = kmax(k, rank_key(-INFINITY, static_cast<uint32_t>(j + e)));
        }
    } else {                                   // scores where the bound says nothing
        for (int j = lo + 8 * lane; j < hi; j += 8 * 64)
            k = kmax(k, exact_chunk<LDT>(row, j, hi, r, inv_t, seed, offset));
    }
    return k;
}

// Grid (rows, parts): workgroup (r, p) takes the p-th contiguous part of row r. parts == 1: it writes
// the row's token. parts > 1 (few rows: one workgroup a row leaves most CUs idle): the parts meet by
// an atomic max of their keys in out[r] itself, which sample_begin_kernel cleared and
// sample_end_kernel turns into the token.
template <int LDT>
__global__ __launch_bounds__(64 * kSampleWaves) void sample_kernel(int64_t* __restrict__ out,
                                                                   const void* __restrict__ logits,
                                                                   const int64_t* __restrict__ rows,
                                                                   const float* __restrict__ temps, int V,
                                                                   uint64_t seed, uint64_t offset) {
    __shared__ unsigned long long winner;
    __shared__ float wave_top[kSampleWaves];
    const int r = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) winner = 0ull;
    const int64_t src = rows ? rows[r] : r;
    const char* row = static_cast<const char*>(logits) + static_cast<size_t>(src) * V * (LDT == CVH_DTYPE_F32 ? 4 : 2);
    const float t = temps ? temps[r] : 0.f;
    // contiguous slice of this wave, a multiple of 8 so a Philox block never straddles slices
    const int slices = kSampleWaves * static_cast<int>(gridDim.y);
    const int slice = ((V + slices * 8 - 1) / (slices * 8)) * 8;
    const int lo = min(V, (static_cast<int>(blockIdx.y) * kSampleWaves + wave) * slice), hi = min(V, lo + slice);
    uint64_t k = t > 0.f ? scan_gumbel<LDT>(row, lo, hi, V, lane, wave, r, 1.0f / fmaxf(t, 1e-5f), seed, offset, wave_top)
                         : scan_greedy<LDT>(row, lo, hi, V, lane);
    k = wave_kmax(k);
    __syncthreads();
    if (lane == 0) atomicMax(&winner, static_cast<unsigned long long>(k));
    __syncthreads();
    if (threadIdx.x == 0) {
        if (gridDim.y == 1) out[r] = key_index(winner);
        else atomicMax(reinterpret_cast<unsigned long long*>(out) + r, winner);
    }
}

__global__ __launch_bounds__(256) void sample_begin_kernel(int64_t* __restrict__ out, int n) {
    const int r = static_cast<int>(blockIdx.x) * 256 + threadIdx.x;
    if (r < n) out[r] = 0;
}
__global__ __launch_bounds__(256) void sample_end_kernel(int64_t* __restrict__ out, int n) {
    const int r = static_cast<int>(blockIdx.x) * 256 + threadIdx.x;
    if (r < n) out[r] = key_index(static_cast<uint64_t>(out[r]));
}

// Parts a row is split into: as many as fill the 256 CUs, each of at least 16384 logits (16 waves of
// two 512-logit loads). The parts meet in out[] by 64-bit atomics, which only this device's own memory is sure
// to take, and clear it first: other memory (pinned host memory, a peer's), or an out[] that is also rows[],
// is written once per row by one workgroup.
bool own_memory(const void* p) {
    hipPointerAttribute_t a{};
    int device = -1;
    if (hipPointerGetAttributes(&a, p) == hipSuccess && hipGetDevice(&device) == hipSuccess)
        return a.type == hipMemoryTypeDevice && a.device == device;
    (void)hipGetLastError();
    return false;
}
int sample_parts(int64_t rows, int vocab, const int64_t* out, const int64_t* row_ids) {
    const int parts = static_cast<int>(std::min<int64_t>(256 / rows, vocab / 16384));
    if (parts <= 1) return 1;
    const uintptr_t o = reinterpret_cast<uintptr_t>(out), i = reinterpret_cast<uintptr_t>(row_ids), n = rows * sizeof(int64_t);
    const bool apart = row_ids == nullptr || o + n <= i || i + n <= o;
    return apart && own_memory(out) ? parts : 1;
}

// ---- token feedback and embedding -------------------------------------------------------------
__global__ __launch_bounds__(256) void feed_tokens_kernel(int64_t* __restrict__ tokens, const int64_t* __restrict__ src,
                                                          const int64_t* __restrict__ prev, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t s = src[i];
    if (s >= 0) tokens[i] = prev[s];
}

// out[t] = table[ids[t]] for 16-bit rows of D elements (D % 8 == 0): one thread per 16 bytes.
__global__ __launch_bounds__(256) void embedding_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ table,
                                                        const int64_t* __restrict__ ids, int64_t T, int D, int64_t V) {
    const int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int per_row = D >> 3;
    if (k >= T * per_row) return;
    const int64_t t = k / per_row;
    const int c = static_cast<int>(k - t * per_row) << 3;
    const int64_t id = ids[t];
    uint4 v = {0u, 0u, 0u, 0u};
    if (id >= 0 && id < V) v = *reinterpret_cast<const uint4*>(table + id * D + c);
    *reinterpret_cast<uint4*>(out + t * D + c) = v;
}

int grid_of(int64_t n, unsigned* g) {
    const int64_t b = (n + 255) / 256;
    if (b > 0x7fffffff) return CVH_ERR_UNSUPPORTED;
    *g = static_cast<unsigned>(b);
    return CVH_OK;
}

int launched() { return hipGetLastError() == hipSuccess ? CVH_OK : CVH_ERR_LAUNCH; }

template <int DT>
int launch_swiglu(void* out, const void* gu, int64_t T, int I, hipStream_t s) {
    using E = typename Elem<DT>::T;
    unsigned g = 0;
    if ((I & 7) == 0) {
        const int64_t n8 = T * (I >> 3);
        if (int rc = grid_of(n8, &g)) return rc;
        if (DT == CVH_DTYPE_BF16 && n8 > kSwigluDirect) {
            const int64_t blocks = (n8 + kSwigluThreads - 1) / kSwigluThreads;
            swiglu_bf16_kernel<<<static_cast<unsigned>(std::min<int64_t>(blocks, kSwigluBlocks)), kSwigluThreads, 0, s>>>(
                    static_cast<uint16_t*>(out), static_cast<const uint16_t*>(gu), n8, I);
        } else {
            swiglu_kernel<DT><<<g, 256, 0, s>>>(static_cast<E*>(out), static_cast<const E*>(gu), n8, I);
        }
    } else {
        if (int rc = grid_of(T * I, &g)) return rc;
        swiglu_scalar_kernel<DT><<<g, 256, 0, s>>>(static_cast<E*>(out), static_cast<const E*>(gu), T * I, I);
    }
    return launched();
}

}  // namespace
}  // namespace cvh

extern "C" int cvh_swiglu(void* out, const void* gate_up, int64_t num_rows, int intermediate, int dtype,
                          cvh_stream_t stream) {
    using namespace cvh;
    if (num_rows < 0 || intermediate <= 0) return CVH_ERR_INVALID_ARG;
    if (num_rows == 0) return CVH_OK;
    if (!out || !gate_up) return CVH_ERR_INVALID_ARG;
    auto s = reinterpret_cast<hipStream_t>(stream);
    switch (dtype) {
        case CVH_DTYPE_BF16: return launch_swiglu<CVH_DTYPE_BF16>(out, gate_up, num_rows, intermediate, s);
        case CVH_DTYPE_F16: return launch_swiglu<CVH_DTYPE_F16>(out, gate_up, num_rows, intermediate, s);
        case CVH_DTYPE_F32: return launch_swiglu<CVH_DTYPE_F32>(out, gate_up, num_rows, intermediate, s);
        default: return CVH_ERR_UNSUPPORTED;
    }
}

extern "C" int cvh_sample_tokens(int64_t* out, const void* logits, int logits_dtype, const int64_t* rows,
                                 const float* temps, int64_t num_rows, int vocab, uint64_t seed, uint64_t offset,
                                 cvh_stream_t stream) {
    using namespace cvh;
    if (num_rows < 0 || vocab <= 0) return CVH_ERR_INVALID_ARG;
    if (num_rows == 0) return CVH_OK;
    if (!out || !logits) return CVH_ERR_INVALID_ARG;
    if (num_rows > 0x7fffffff) return CVH_ERR_UNSUPPORTED;
    auto s = reinterpret_cast<hipStream_t>(stream);
    if (logits_dtype != CVH_DTYPE_F32 && logits_dtype != CVH_DTYPE_BF16) return CVH_ERR_UNSUPPORTED;
    const int parts = sample_parts(num_rows, vocab, out, rows);
    const dim3 grid(static_cast<unsigned>(num_rows), static_cast<unsigned>(parts));
    const int n = static_cast<int>(num_rows);
    if (parts > 1) sample_begin_kernel<<<(n + 255) / 256, 256, 0, s>>>(out, n);
    if (logits_dtype == CVH_DTYPE_F32)
        sample_kernel<CVH_DTYPE_F32><<<grid, 64 * kSampleWaves, 0, s>>>(out, logits, rows, temps, vocab, seed, offset);
    else
        sample_kernel<CVH_DTYPE_BF16><<<grid, 64 * kSampleWaves, 0, s>>>(out, logits, rows, temps, vocab, seed, offset);
    if (parts > 1) sample_end_kernel<<<(n + 255) / 256, 256, 0, s>>>(out, n);
    return launched();
}

extern "C" int cvh_feed_tokens(int64_t* tokens, const int64_t* src, const int64_t* prev, int64_t n,
                               cvh_stream_t stream) {
    using namespace cvh;
    if (n < 0) return CVH_ERR_INVALID_ARG;
    if (n == 0) return CVH_OK;
    if (!tokens || !src || !prev) return CVH_ERR_INVALID_ARG;
    unsigned g = 0;
    if (int rc = grid_of(n, &g)) return rc;
    feed_tokens_kernel<<<g, 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(tokens, src, prev, n);
    return launched();
}

extern "C" int cvh_embedding(void* out, const void* table, const int64_t* ids, int64_t num_tokens, int dim,
                             int64_t vocab, cvh_stream_t stream) {
    using namespace cvh;
    if (num_tokens < 0 || dim <= 0 || vocab <= 0) return CVH_ERR_INVALID_ARG;
    if (num_tokens == 0) return CVH_OK;
    if (!out || !table || !ids) return CVH_ERR_INVALID_ARG;
    if ((dim & 7) != 0) return CVH_ERR_UNSUPPORTED;
    unsigned g = 0;
    if (int rc = grid_of(num_tokens * (dim >> 3), &g)) return rc;
    embedding_kernel<<<g, 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(
            static_cast<uint16_t*>(out), static_cast<const uint16_t*>(table), ids, num_tokens, dim, vocab);
    return launched();
}
