// Which projections the few-row kernels (gemv.hip) take; the decode runner asks before it plans a layer.
#pragma once

#include <stdint.h>

namespace cvh {

// Rows: every wave norms them all again, which still costs less than the launches that it saves (28-layer step,
// Qwen3-0.6B, contexts 100 to 1024: 1 / 2 / 3 / 4 rows 902 / 1013 / 1081 / 1097 us, by the general path 1359 / 1495 /
// 1516 / 1558; 5 rows take that one, 1504). More than four are not measured.
constexpr int kMvMaxRows = 4;
// K in whole 512-element turns of a wave: up to 2048 where the input is normed (a wave holds four columns and
// the rows in registers), up to 4096 for the residual projections (one column); N in whole workgroups of 16
// columns.
inline bool gemv_ok(int64_t M, int64_t N, int64_t K, int64_t max_k) {
    return M >= 1 && M <= kMvMaxRows && N > 0 && N % 16 == 0 && K > 0 && K % 512 == 0 && K <= max_k;
}
constexpr int64_t kMvNormMaxK = 2048, kMvResidMaxK = 4096;

}  // namespace cvh
