// Which projections the few-row kernels (gemv.hip) take; the decode runner asks before it plans a layer.
#pragma once

#include <stdint.h>

namespace cvh {

constexpr int kMvMaxRows = 4;
// K in whole 512-element turns of a wave: up to 2048 where the input is normed or two columns share a wave,
// up to 4096 for the residual projections; N in whole workgroups of 16 columns.
inline bool gemv_ok(int64_t M, int64_t N, int64_t K, int64_t max_k) {
    return M >= 1 && M <= kMvMaxRows && N > 0 && N % 16 == 0 && K > 0 && K % 512 == 0 && K <= max_k;
}
constexpr int64_t kMvNormMaxK = 2048, kMvResidMaxK = 4096;

}  // namespace cvh
