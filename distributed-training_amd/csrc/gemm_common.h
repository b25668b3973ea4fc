// Shared by the GEMM kernels (gemm.hip, gemm_direct.hip): the MFMA shapes, the
// launch arguments, the fused epilogue of one element, the block-to-tile order
// and the column sums' last step.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.h"
#include "gelu.h"

namespace dtmi {

template <typename T>
struct MF;

template <>
struct MF<float> {
  static constexpr int MT = 32, G = 2, VEC = 4, NACC = 16;
  typedef float acc_t __attribute__((ext_vector_type(16)));
  typedef float vec_t __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
  }
  // result register i of lane group g holds row (8*(i/4) + 4*g + i%4), column lane%32
  static __device__ __forceinline__ int row(int i, int g) { return 8 * (i / 4) + 4 * g + (i % 4); }
};

template <>
struct MF<double> {
  static constexpr int MT = 16, G = 4, VEC = 2, NACC = 4;
  typedef double acc_t __attribute__((ext_vector_type(4)));
  typedef double vec_t __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // result register i of lane group g holds row (g + 4*i), column lane%16
  static __device__ __forceinline__ int row(int i, int g) { return g + 4 * i; }
};

struct GemmArgs {
  const void* A;
  const void* B;
  void* C;
  const void* bias;
  void* ws;  // split-K partials [splits][batch][M][N] (NULL when not split)
  int64_t M, N, K, lda, ldb, ldc;
  int64_t sA, sB, sC;  // batch strides (elements)
  int64_t k_per_split;
  int tiles_m, tiles_n;
  int accumulate;
  // 64 x 64 tile: accumulators added into a second set after every this many
  // groups of k-tiles (0: one chain over the whole k range)
  int fold_groups;
  // Epilogue fusions (applied after the bias, in this order):
  const void* addend;  // residual: v = addend[m, n] + v   (row stride ldc)
  int epi;             // kEpiGeluFwd: aux = gelu(v), C keeps v; kEpiGeluBwd: C = gelu'(aux) * v
  void* aux;           // [M, N] with row stride ldc
  // Column sums of B over k (the bias gradient of dW = X^T dY: db = sum over
  // rows of dY), taken by the blocks of the first row of tiles from the B
  // tiles already in LDS. Unbatched only. With split-K each split's sums go to
  // colsum_ws[split][n] and the reduction kernel adds them in split order.
  void* colsum;
  void* colsum_ws;
  int colsum_accumulate;
};

// k-tile: 16 floats or 8 doubles
template <typename T>
constexpr int kBKT = sizeof(T) == 4 ? 16 : 8;

constexpr int kEpiNone = 0, kEpiGeluFwd = 1, kEpiGeluBwd = 2;

// The fused epilogue of one output element v (the k-sum of row m, column n):
// bias, residual, accumulate, GELU -- the operation order of the unfused
// graph (Linear adds its bias, then the residual add, then GELU / its
// backward as dtrain/autograd.py:133-144 computes them).
template <typename T>
__device__ __forceinline__ void epilogue_store(const GemmArgs& a, T* __restrict__ C, int64_t ldc, int64_t m,
                                               int64_t n, T v, int64_t batch) {
  if (a.bias) v = v + ((const T*)a.bias)[n];
  const int64_t o = m * ldc + n;
  if (a.addend) v = ((const T*)a.addend)[batch * a.sC + o] + v;
  if (a.accumulate) v = C[o] + v;
  if (a.epi == kEpiGeluFwd) {
    ((T*)a.aux)[batch * a.sC + o] = gelu_f<T>(v);
  } else if (a.epi == kEpiGeluBwd) {
    v = gelu_b<T>(((const T*)a.aux)[batch * a.sC + o], v);
  }
  C[o] = v;
}

__device__ __forceinline__ void tile_coords_of(const GemmArgs& a, int t, int& tm, int& tn) {
  const int nt = a.tiles_m * a.tiles_n;
  if ((nt & 7) == 0) t = (t & 7) * (nt >> 3) + (t >> 3);  // contiguous tile range per XCD
  constexpr int GROUP = 8;
  const int per_group = GROUP * a.tiles_n;
  const int group = t / per_group;
  const int first_m = group * GROUP;
  const int gsz = a.tiles_m - first_m < GROUP ? a.tiles_m - first_m : GROUP;
  const int r = t - group * per_group;
  tm = first_m + r % gsz;
  tn = r / gsz;
}
__device__ __forceinline__ void tile_coords(const GemmArgs& a, int& tm, int& tn) {
  tile_coords_of(a, (int)blockIdx.x, tm, tn);
}

// The column sum of one B column over this block's k range: to colsum (or
// added to it), or, with split-K, to the split's row of colsum_ws.
template <typename T>
__device__ __forceinline__ void finish_colsum(const GemmArgs& a, double csum, int64_t n, int split) {
  if (n >= a.N) return;
  if (a.colsum_ws) {
    ((T*)a.colsum_ws)[(int64_t)split * a.N + n] = (T)csum;
  } else {
    T* cs = (T*)a.colsum;
    cs[n] = a.colsum_accumulate ? cs[n] + (T)csum : (T)csum;
  }
}

}  // namespace dtmi
