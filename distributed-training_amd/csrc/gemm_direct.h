// The small-product GEMM kernel's launch (gemm_direct.hip).
#pragma once

#include "gemm_common.h"

namespace dtmi {

// Launches C = A B with a's epilogue and column sums, a.k_per_split of k per wave
// (K >= 1, at most kDirectMaxWaves<T> waves; leading dimensions below 2^24 bytes,
// any alignment). a.ws and the tiles are set here.
template <typename T>
constexpr int kDirectMaxWaves = sizeof(T) == 4 ? 16 : 8;  // 64 KB of partial tiles
template <typename T>
constexpr int kDirectBatch = sizeof(T) == 4 ? 32 : 16;  // k per batch of loads
template <typename T>
void launch_gemm_direct(GemmArgs a, int64_t batch, int akc, int bkc);

}  // namespace dtmi
