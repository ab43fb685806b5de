// Projections of up to four rows on gfx950: Y[M][N] = X[M][K] . W[N][K]^T with one wave per few output
// columns (bf16 in, fp32 accumulation with v_dot2_f32_bf16, bf16 out), and the layer boundaries of a
// decode step fused at their rounding points: an input that is the RMSNorm of the residual, a
// residual add, SwiGLU.
//
// At one row a decode layer reads 31 MB of weights and does little else, so what counts is how many
// bytes are in flight and how many launches the layer takes. The matrix-core kernels give 16 columns to a
// workgroup: 64 workgroups for a 1024-column projection, each waiting out its loads chunk by chunk. Here a
// wave owns CW columns and requests all of their K * CW weights at once (4 to 8 KB), so 256 workgroups of 4
// waves have the whole matrix in flight. Lane l holds elements 8l + 512i .. +8 of every row and column, the
// same elements that norm_row gives it, so a wave norms its input rows in registers to the bits of the
// standalone kernel; sums over K are per lane in index order, then an xor butterfly over the 64 lanes.
// One row, Qwen3-0.6B shapes, weights from HBM (kernel times): QKV 3.8 (norm) + 4.0 -> 3.6 us, o_proj 5.9 +
// 3.8 (add + norm) -> 3.1, gate/up 6.4 -> 4.5, down 5.9 + 3.8 -> 3.1; graph of 28 layers 1359 -> 902 us.
#include <hip/hip_runtime.h>

#include "cvh_device.h"
#include "gemv.h"

namespace cvh {
namespace {

enum { kMvStore = 0, kMvResid = 1, kMvSwiglu = 2 };

struct MvArgs {
    uint16_t* y;               // kMvStore [M][N]; kMvResid: the residual [M][N], in place; kMvSwiglu: act [M][N/2]
    const uint16_t* x;         // [M][K]
    const uint16_t* w;         // [N][K] (kMvSwiglu: gate/up rows interleaved by 16)
    const uint16_t* gain;      // NORM: [K]
    float eps;
    int M, N;
};

typedef uint32_t mv_u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float mv_dot(const mv_u32x4& a, const mv_u32x4& b, float c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t aj = a[j], bj = b[j];       // (a bit cast of a vector's element takes element 0)
        c = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16_pair_t, aj), __builtin_bit_cast(bf16_pair_t, bj), c,
                                            false);
    }
    return c;
}

// MB rows per workgroup (blockIdx.y), CW columns per wave (kMvSwiglu: CW / 2 outputs, their gate and up
// columns), K = 512 * NI.
template <int MB, int CW, int NI, int EPI, bool NORM>
__device__ __forceinline__ void gemv_body(const MvArgs& a) {
    constexpr int K = 512 * NI;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = (static_cast<int>(blockIdx.x) * 4 + wave) * CW;       // first column of the wave
    const int m0 = static_cast<int>(blockIdx.y) * MB;
    auto column = [&](int c) {       // kMvSwiglu: output j = first/2 + c/2, gate (c even) then up
        if constexpr (EPI == kMvSwiglu) {
            const int j = (first >> 1) + (c >> 1);
            return (j >> 4) * 32 + (j & 15) + (c & 1) * 16;
        } else {
            return first + c;
        }
    };
    mv_u32x4 wv[CW][NI];
#pragma unroll
    for (int c = 0; c < CW; ++c) {
        const uint16_t* wp = a.w + static_cast<size_t>(column(c)) * K + lane * 8;
#pragma unroll
        for (int i = 0; i < NI; ++i) wv[c][i] = __builtin_nontemporal_load(reinterpret_cast<const mv_u32x4*>(wp + 512 * i));
    }
    mv_u32x4 xv[MB][NI];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const uint16_t* xp = a.x + static_cast<size_t>(min(m0 + m, a.M - 1)) * K + lane * 8;     // rows past M: the last
#pragma unroll
        for (int i = 0; i < NI; ++i) xv[m][i] = *reinterpret_cast<const mv_u32x4*>(xp + 512 * i);
    }
    // the residual of this wave's columns, one (row, column) per lane
    const int em = lane / CW, ec = lane % CW;
    const bool mine = lane < MB * CW && m0 + em < a.M;
    uint16_t* yp = a.y + static_cast<size_t>(m0 + em) * a.N + first + ec;
    float res = 0.f;
    if constexpr (EPI == kMvResid) res = mine ? bf16_bits_to_f32(*yp) : 0.f;
    if constexpr (NORM) {
        mv_u32x4 gv[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) gv[i] = *reinterpret_cast<const mv_u32x4*>(a.gain + lane * 8 + 512 * i);
#pragma unroll
        for (int m = 0; m < MB; ++m) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float lo = __uint_as_float(xv[m][i][j] << 16), hi = __uint_as_float(xv[m][i][j] & 0xffff0000u);
                    ss = ss + lo * lo;
                    ss = ss + hi * hi;
                }
            ss = xor_sum<64>(ss);
            const float inv = 1.0f / __builtin_sqrtf(ss / static_cast<float>(K) + a.eps);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float lo = __uint_as_float(xv[m][i][j] << 16) * inv, hi = __uint_as_float(xv[m][i][j] & 0xffff0000u) * inv;
                    round_bf16x2(lo, hi);
                    xv[m][i][j] = pack_bf16x2(lo * __uint_as_float(gv[i][j] << 16), hi * __uint_as_float(gv[i][j] & 0xffff0000u));
                }
        }
    }
    float acc[MB][CW];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < NI; ++i) s = mv_dot(wv[c][i], xv[m][i], s);
            acc[m][c] = xor_sum<64>(s);
        }
    // lane (m, c) stores its value (kMvSwiglu: the even columns' lanes)
    float v = acc[0][0], u = 0.f;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            if (lane == m * CW + c) v = acc[m][c];
            if constexpr (EPI == kMvSwiglu)
                if (lane == m * CW + c && (c & 1) == 0) u = acc[m][c + 1];
        }
    if (!mine) return;
    if constexpr (EPI == kMvStore) {
        *yp = f32_to_bf16_bits(v);
    } else if constexpr (EPI == kMvResid) {
        *yp = f32_to_bf16_bits(res + round_bf16(v));
    } else if ((ec & 1) == 0) {
        a.y[static_cast<size_t>(m0 + em) * (a.N >> 1) + ((first + ec) >> 1)] =
                f32_to_bf16_bits(silu_mul<CVH_DTYPE_BF16>(round_bf16(v), round_bf16(u)));
    }
}

template <int MB, int CW, int NI, int EPI, bool NORM>
__global__ __launch_bounds__(256) void gemv_kernel(MvArgs a) {
    gemv_body<MB, CW, NI, EPI, NORM>(a);
}

// Columns per wave: 4 where the input is normed (the norm is repeated per wave: 1024 waves for a 4096-column
// QKV projection, 1536 for the 3072 outputs of gate/up); 1 for the residual projections, whose 1024
// columns then still make 256 workgroups.
template <int MB, int CW, int NI, int EPI, bool NORM>
int launch_gemv(const MvArgs& a, hipStream_t s) {
    gemv_kernel<MB, CW, NI, EPI, NORM><<<dim3(a.N / (4 * CW), (a.M + MB - 1) / MB), 256, 0, s>>>(a);
    return hipGetLastError() == hipSuccess ? CVH_OK : CVH_ERR_LAUNCH;
}
template <int CW, int NI, int EPI, bool NORM>
int launch_rows(const MvArgs& a, hipStream_t s) {
    if (a.M == 1) return launch_gemv<1, CW, NI, EPI, NORM>(a, s);
    if (a.M == 2) return launch_gemv<2, CW, NI, EPI, NORM>(a, s);
    return launch_gemv<4, CW, NI, EPI, NORM>(a, s);
}
template <int CW, int EPI, bool NORM, int MAXNI, int NI = 1>
int launch_k(int ni, const MvArgs& a, hipStream_t s) {
    if (ni == NI) return launch_rows<CW, NI, EPI, NORM>(a, s);
    if constexpr (NI < MAXNI) return launch_k<CW, EPI, NORM, MAXNI, NI + 1>(ni, a, s);
    return CVH_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace cvh

extern "C" int cvh_gemv_bf16_norm(void* y, const void* x, const void* gain, double eps, const void* w, int64_t M, int N,
                                  int K, cvh_stream_t stream) {
    using namespace cvh;
    if (M < 0 || N <= 0 || K <= 0) return CVH_ERR_INVALID_ARG;
    if (M == 0) return CVH_OK;
    if (!y || !x || !gain || !w) return CVH_ERR_INVALID_ARG;
    if (!gemv_ok(M, N, K, kMvNormMaxK)) return CVH_ERR_UNSUPPORTED;
    const MvArgs a{static_cast<uint16_t*>(y), static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w),
                   static_cast<const uint16_t*>(gain), static_cast<float>(eps), static_cast<int>(M), N};
    return launch_k<4, kMvStore, true, kMvNormMaxK / 512>(K / 512, a, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int cvh_gemv_bf16_residual(void* resid, const void* x, const void* w, int64_t M, int N, int K,
                                      cvh_stream_t stream) {
    using namespace cvh;
    if (M < 0 || N <= 0 || K <= 0) return CVH_ERR_INVALID_ARG;
    if (M == 0) return CVH_OK;
    if (!resid || !x || !w) return CVH_ERR_INVALID_ARG;
    if (!gemv_ok(M, N, K, kMvResidMaxK)) return CVH_ERR_UNSUPPORTED;
    const MvArgs a{static_cast<uint16_t*>(resid), static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w), nullptr,
                   0.f, static_cast<int>(M), N};
    return launch_k<1, kMvResid, false, kMvResidMaxK / 512>(K / 512, a, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int cvh_gemv_bf16_norm_swiglu(void* act, const void* x, const void* gain, double eps, const void* w, int64_t M,
                                         int I, int K, cvh_stream_t stream) {
    using namespace cvh;
    if (M < 0 || I <= 0 || K <= 0) return CVH_ERR_INVALID_ARG;
    if (M == 0) return CVH_OK;
    if (!act || !x || !gain || !w) return CVH_ERR_INVALID_ARG;
    if (I > (1 << 29) || I % 16 || !gemv_ok(M, 2 * I, K, kMvNormMaxK)) return CVH_ERR_UNSUPPORTED;
    const MvArgs a{static_cast<uint16_t*>(act), static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(w),
                   static_cast<const uint16_t*>(gain), static_cast<float>(eps), static_cast<int>(M), 2 * I};
    return launch_k<4, kMvSwiglu, true, kMvNormMaxK / 512>(K / 512, a, reinterpret_cast<hipStream_t>(stream));
}
