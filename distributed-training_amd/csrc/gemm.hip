// Dense contractions on the MFMA matrix cores: C = sum_k A(m,k) B(k,n) (+ bias)
// in float32 (v_mfma_f32_32x32x2_f32) and float64 (v_mfma_f64_16x16x4_f64).
//
// Behind dtrain's matmul node (dtrain/autograd.py:102-109) and Linear
// (dtrain/nn.py:58-65): forward Y = X W (+ b), dX = dY W^T, dW = X^T dY.
// Row-major operands in either orientation:
//   A "KC": A(m,k) = A[m*lda + k]  (X, dY)      A "MC": A(m,k) = A[k*lda + m]  (X^T)
//   B "NC": B(k,n) = B[k*ldb + n]  (W, dY)      B "KC": B(k,n) = B[n*ldb + k]  (W^T)
//
// Tiling. 256 threads = 4 waves in a 2x2 grid; block tile 128x128; k-tile
// 16 floats or 8 doubles; MFMA tiles of 32x32 (float32) or 16x16 (float64).
// Each operand tile is staged in LDS in its global orientation (global -> LDS
// is a straight 16-byte vector copy, fully coalesced along the contiguous
// dimension), with one barrier per k-tile and the next tiles' global loads in
// flight during the MFMAs (rows past the matrix edge clamped onto the last row).
//   gemm_dma_kernel: the loads go straight into LDS (global_load_lds) through
//     three stages, in swizzled layouts that keep the fragment reads
//     conflict-free; a wave-uniform base advanced by scalar adds and fixed lane
//     offsets, so the main loop has no vector instruction but the MFMAs. 16-byte
//     granular operands (every GPT-2 GEMM, in float32 and float64) take 16 bytes
//     per lane, others 4: the vocabulary head's products at 50257 columns ran
//     element by element through registers at 64 to 107 TFLOP/s, and run at 136 to
//     140 (forward 2961 -> 2256 us, dX 4948 -> 2321, dW 3301 -> 2334).
//   gemm_kernel (leading dimensions of 2^24 bytes and more): registers -> LDS,
//     double-buffered.
//   gemm_x6_kernel (float32 when dtmi_set_gemm_math selects the split-bf16
//     arithmetic, aligned operands): each operand split exactly into three
//     bf16 parts on the way into LDS, six partial products on the bf16 MFMA
//     (its own section below).
// (256x128 and 128x256 tiles, 32-wide k-tiles, a two-tile register prefetch
// and AGPR accumulators measured no faster on the GPT-2 shapes.)
//
// MFMA k-slots. An MFMA takes k in lane groups g = lane / MT (2 groups of 32
// lanes for 32x32x2, 4 groups of 16 for 16x16x4). Within each 8-wide k chunk,
// step s of group g uses k = chunk + VEC*g + s (VEC = 4 floats or 2 doubles),
// the same permutation for A and B (a permutation of the reduction index does
// not change the sum's terms). With it a k-contiguous LDS tile gives a lane
// its VEC k-values with one 16-byte ds_read, and an mn-contiguous LDS tile is
// read with conflict-free 4/8-byte reads (row pads chosen so the lane groups
// fall in different LDS banks).
//
// Grid. Tiles are enumerated group-of-8-rows first (L2 reuse of B panels) and
// the linear block index is remapped so each of the 8 XCDs (blocks are dealt
// to XCDs round-robin) works on a contiguous range of tiles and shares its L2.
// Small tile counts with long K are split along K; the split partials are
// summed in split order by a second kernel (deterministic, no atomics).
#include "common.h"
#include "bufrsrc.h"
#include "gelu.h"
#include "gemm_common.h"
#include "gemm_direct.h"
#include "rowln.h"

namespace dtmi {

// gemm_f32.hip, gemm_f32_64.hip, gemm_f32_256.hip, gemm_f64.hip, gemm_f64_64.hip, gemm_x6.hip
template <typename T, int BM, int BN>
void launch_layout(const GemmArgs& a, dim3 grid, int akc, int bkc, bool veca, bool vecb, bool dma);
void launch_x6(const GemmArgs& a, dim3 grid, int akc, int bkc);

// Sum of the split-K partials in split order 0, 1, ..., S-1, then the
// epilogue. PLAIN (bias only): VEC consecutive columns per thread.
template <typename T, bool PLAIN, int VEC>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(GemmArgs a, const T* __restrict__ ws, int splits,
                                                             int64_t batch) {
  const int64_t M = a.M, N = a.N;
  const int64_t total = batch * M * N;
  const int64_t nvec = total / VEC;  // VEC divides N
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const T* __restrict__ bias = (const T*)a.bias;
  if (a.colsum_ws) {  // column sums of the splits, in split order
    T* cs = (T*)a.colsum;
    const T* w = (const T*)a.colsum_ws;
    for (int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; n < N; n += stride) {
      T v = w[n];
      for (int s = 1; s < splits; ++s) v = v + w[(int64_t)s * N + n];
      cs[n] = a.colsum_accumulate ? cs[n] + v : v;
    }
  }
  for (int64_t iv = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; iv < nvec; iv += stride) {
    const int64_t idx = iv * VEC;
    const int64_t b = idx / (M * N);
    const int64_t rem = idx - b * M * N;
    const int64_t m = rem / N, n = rem - m * N;
    T* C = (T*)a.C + b * a.sC;
    if (VEC > 1) {  // 16-byte vectors: every operand is aligned (checked by the host)
      typedef T vt __attribute__((ext_vector_type(VEC)));
      vt v = *reinterpret_cast<const vt*>(ws + idx);
      // four partials loaded at a time, added in split order
      int s = 1;
      for (; s + 3 < splits; s += 4) {
        vt t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = *reinterpret_cast<const vt*>(ws + (int64_t)(s + u) * total + idx);
#pragma unroll
        for (int u = 0; u < 4; ++u) v = v + t[u];
      }
      for (; s < splits; ++s) v = v + *reinterpret_cast<const vt*>(ws + (int64_t)s * total + idx);
      if (bias) v = v + *reinterpret_cast<const vt*>(bias + n);
      const int64_t o = m * a.ldc + n;
      if (!PLAIN) {  // the epilogue_store sequence, VEC elements at a time
        if (a.addend) v = *reinterpret_cast<const vt*>((const T*)a.addend + b * a.sC + o) + v;
        if (a.accumulate) v = *reinterpret_cast<const vt*>(C + o) + v;
        if (a.epi == kEpiGeluFwd) {
          vt y;
#pragma unroll
          for (int e = 0; e < VEC; ++e) y[e] = gelu_f<T>(v[e]);
          *reinterpret_cast<vt*>((T*)a.aux + b * a.sC + o) = y;
        } else if (a.epi == kEpiGeluBwd) {
          const vt x = *reinterpret_cast<const vt*>((const T*)a.aux + b * a.sC + o);
#pragma unroll
          for (int e = 0; e < VEC; ++e) v[e] = gelu_b<T>(x[e], v[e]);
        }
      }
      *reinterpret_cast<vt*>(C + o) = v;
      continue;
    }
    T v[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[e] = ws[idx + e];
    for (int s = 1; s < splits; ++s) {
      const T* w = ws + (int64_t)s * total + idx;
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[e] = v[e] + w[e];
    }
    if (PLAIN) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) C[m * a.ldc + n + e] = bias ? v[e] + bias[n + e] : v[e];
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) epilogue_store<T>(a, C, a.ldc, m, n + e, v[e], b);
    }
  }
}

// Row dots of a float32 product whose rows are H = N / 64 groups of 64
// columns -- the attention output's gradient dO = dY W^T of the projection
// that reads the attention output X = O -- with X: rowdot[(b H + h) T + t] =
// sum_d C[m, 64 h + d] X[m, 64 h + d] for row m = b T + t, the rowsum(dO * O)
// term of the attention backward. Summed as the attention backward's own
// row pass sums it (four products in order, then a 16-lane butterfly), so the
// bits are that pass's. splitk_rowdot_kernel also forms C as the plain
// split-K sum (splitk_reduce_kernel's order); rowdot64_kernel reads a finished
// C. 16 consecutive threads cover one (row, group): N % 64 == 0.
__device__ __forceinline__ void rowdot_group(float d, int64_t idx, int64_t N, int64_t T, float* __restrict__ rowdot) {
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) d += __shfl_xor(d, off, 16);
  if ((threadIdx.x & 15) == 0) {
    const int64_t m = idx / N, h = (idx - m * N) / 64, b = m / T, t = m - b * T;
    rowdot[(b * (N / 64) + h) * T + t] = d;
  }
}

__global__ void __launch_bounds__(256) splitk_rowdot_kernel(GemmArgs a, const float* __restrict__ ws, int splits,
                                                             const float* __restrict__ X, float* __restrict__ rowdot,
                                                             int64_t T) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const int64_t N = a.N, total = a.M * N, nvec = total / 4;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  float* C = (float*)a.C;
  for (int64_t iv = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; iv < nvec; iv += stride) {
    const int64_t idx = iv * 4;
    // X and the first two partials in flight together
    const f4 o = *reinterpret_cast<const f4*>(X + idx);
    f4 v = *reinterpret_cast<const f4*>(ws + idx);
    const f4 p1 = *reinterpret_cast<const f4*>(ws + total + idx);  // splits >= 2
    v = v + p1;
    int s = 2;
    for (; s + 3 < splits; s += 4) {
      f4 t[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) t[u] = *reinterpret_cast<const f4*>(ws + (int64_t)(s + u) * total + idx);
#pragma unroll
      for (int u = 0; u < 4; ++u) v = v + t[u];
    }
    for (; s < splits; ++s) v = v + *reinterpret_cast<const f4*>(ws + (int64_t)s * total + idx);
    *reinterpret_cast<f4*>(C + idx) = v;
    rowdot_group(((o[0] * v[0] + o[1] * v[1]) + o[2] * v[2]) + o[3] * v[3], idx, N, T, rowdot);
  }
}

__global__ void __launch_bounds__(256) rowdot64_kernel(const float* __restrict__ C, const float* __restrict__ X,
                                                        float* __restrict__ rowdot, int64_t M, int64_t N, int64_t T) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const int64_t nvec = M * N / 4;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t iv = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; iv < nvec; iv += stride) {
    const int64_t idx = iv * 4;
    const f4 v = *reinterpret_cast<const f4*>(C + idx);
    const f4 o = *reinterpret_cast<const f4*>(X + idx);
    rowdot_group(((o[0] * v[0] + o[1] * v[1]) + o[2] * v[2]) + o[3] * v[3], idx, N, T, rowdot);
  }
}

// Split-K sum, bias and residual of an output row, then the LayerNorm of the
// finished row, in one pass: one wave per row, the row in registers. The
// output element is (((p_0 + p_1) + ...) + bias) then residual + that -- the
// reduction kernel's and epilogue's order -- and the LayerNorm is the shared
// row code of the LayerNorm kernel, so C, ln_out, mean and rstd are the bits
// the separate kernels give. 16-byte aligned rows, unbatched. S2: exactly
// two partials (the common split), loaded with no stand-in re-reads.
template <typename T, int NV, int VW, bool S2>
__global__ void __launch_bounds__(256) splitk_ln_kernel(GemmArgs a, const T* __restrict__ ws, int splits,
                                                         T* __restrict__ hout, T* __restrict__ mean,
                                                         T* __restrict__ rstd, const T* __restrict__ lw,
                                                         const T* __restrict__ lb, T eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t M = a.M;
  const int cols = (int)a.N;
  if (row >= M) return;
  const int64_t total = M * a.N;
  const T* bias = (const T*)a.bias;
  const T* add = (const T*)a.addend;
  T* C = (T*)a.C;
  // every load of the row is issued before the first add, from addresses
  // that are always valid (a missing split, bias or residual re-reads the
  // first partial and is then left out), so no load waits behind a branch
  constexpr int SP = S2 ? 2 : (NV * VW <= 16 ? 4 : (NV * VW <= 32 ? 2 : 1));
  if (S2) splits = 2;
  T pv[SP][NV][VW], bv[NV][VW], rv[NV][VW];
  const T* bsrc = bias ? bias : ws;
  const T* rsrc = add ? add + row * a.ldc : ws + row * a.N;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = VW * lane + 64 * VW * j;
    const int cc = c < cols ? c : 0;
    const int64_t idx = row * a.N + cc;
#pragma unroll
    for (int sp = 0; sp < SP; ++sp) load_vec<T, VW>(pv[sp][j], ws + (int64_t)(sp < splits ? sp : 0) * total + idx);
    load_vec<T, VW>(bv[j], bsrc + cc);
    load_vec<T, VW>(rv[j], rsrc + cc);
  }
  T xv[NV][VW];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = VW * lane + 64 * VW * j;
    T v[VW];
#pragma unroll
    for (int e = 0; e < VW; ++e) v[e] = pv[0][j][e];
#pragma unroll
    for (int sp = 1; sp < SP; ++sp)
      if (sp < splits)
#pragma unroll
        for (int e = 0; e < VW; ++e) v[e] = v[e] + pv[sp][j][e];
    if (c < cols) {
      for (int sp = SP; sp < splits; ++sp) {  // more splits than held in registers
        T t[VW];
        load_vec<T, VW>(t, ws + (int64_t)sp * total + row * a.N + c);
#pragma unroll
        for (int e = 0; e < VW; ++e) v[e] = v[e] + t[e];
      }
    }
    if (bias)
#pragma unroll
      for (int e = 0; e < VW; ++e) v[e] = v[e] + bv[j][e];
    if (add)
#pragma unroll
      for (int e = 0; e < VW; ++e) v[e] = rv[j][e] + v[e];
    if (c < cols) {
      store_vec<T, VW>(C + row * a.ldc + c, v);
#pragma unroll
      for (int e = 0; e < VW; ++e) xv[j][e] = v[e];
    } else {
#pragma unroll
      for (int e = 0; e < VW; ++e) xv[j][e] = T(0);
    }
  }
  ln_row_fwd<T, NV, VW>(xv, cols, lane, lw, lb, eps, hout + row * cols, mean + row, rstd + row);
}

// float32 GEMM arithmetic: DTMI_GEMM_MATH_F32 (float32 MFMA) or
// DTMI_GEMM_MATH_BF16X6 (exact 3-way bf16 split, 6 bf16 MFMA products).
static int g_gemm_math = DTMI_GEMM_MATH_F32;

struct EpiArgs {
  const void* addend = nullptr;
  int epi = kEpiNone;
  void* aux = nullptr;
  void* colsum = nullptr;  // column sums of B (length N), unbatched
  int colsum_accumulate = 0;
  // Split-K partials left for the consumer: when the chooser takes between 2
  // and parts_max splits, the raw partials go to parts_out ([splits][M][N],
  // unbatched, no bias or epilogue) with no sum pass and *parts_n = splits;
  // otherwise C is written as usual and *parts_n = 1.
  void* parts_out = nullptr;
  int parts_max = 0;
  int* parts_n = nullptr;
  // float32 row dots with X per 64-column group (see splitk_rowdot_kernel)
  const void* rowdot_x = nullptr;
  void* rowdot_out = nullptr;
  int64_t rowdot_T = 1;
  // LayerNorm of the finished output rows (after bias and residual):
  // ln_out = layer_norm(C; ln_w, ln_b, ln_eps), with the row mean and rstd
  void* ln_out = nullptr;
  void* ln_mean = nullptr;
  void* ln_rstd = nullptr;
  const void* ln_w = nullptr;
  const void* ln_b = nullptr;
  double ln_eps = 1e-5;
};

// K splits. A grid of b blocks on C CUs runs ceil(b / C) rounds, so its
// useful fraction is b / (C * ceil(b / C)); take the fewest splits (each
// keeping >= 256 of K) that reach 90 % of rounds, else the best found. A grid
// of fewer than ~2 blocks per CU leaves one wave per SIMD, which cannot hide
// its own latencies: it counts 15 % less (measured: the 768 x 768 x 8192
// weight gradient ran at 114 TFLOP/s on 252 blocks).
static int choose_splits(int64_t tiles, int64_t batch, int64_t K, int64_t cus) {
  int splits = 1;
  double e_best = 0.0;
  for (int sp = 1; sp <= 16; ++sp) {
    if (sp > 1 && K / sp < 256) break;
    const int64_t blocks = tiles * batch * sp;
    double eff = (double)blocks / (double)(cus * cdiv(blocks, cus));
    if (10 * blocks < 19 * cus) eff *= 0.85;
    if (eff > e_best + 1e-9) {
      e_best = eff;
      splits = sp;
    }
    if (eff >= 0.9) break;
  }
  return splits;
}

// Block tile of the aligned float32 kernel: 256 x 128 when every block still
// gets a long k range (>= 1024) and the grid covers the CUs, else 128 x 128.
// The larger tile moves 25 % fewer bytes per MFMA through the loads and LDS
// but has half the blocks; on the GPT-2 shapes it wins for the long-K
// products (dW, the vocabulary head's dX and dW) and loses on K = 768. When
// the larger tile needs a K split and the smaller one fills whole rounds
// without one, the smaller one is taken: no partials, no sum pass.
static void pick_tile(int64_t M, int64_t N, int64_t K, int64_t batch, int64_t cus, int& bm, int& bn) {
  bm = bn = 128;
  if (M < 256) return;
  const int64_t tiles = cdiv(M, 256) * cdiv(N, 128);
  const int sp = choose_splits(tiles, batch, K, cus);
  if (tiles * batch * sp >= cus && K / sp >= 1024) bm = 256;
  if (bm == 256 && sp > 1) {
    const int64_t t128 = cdiv(M, 128) * cdiv(N, 128);
    if (choose_splits(t128, batch, K, cus) == 1 && t128 * batch % cus == 0) bm = 128;
  }
}

// Estimated time of a plan in SIMD cycles, to compare the 64 x 64 tile and the
// small-product kernel with the 128-wide tiles. A 32 x 32 piece of the output
// takes 32 MFMA cycles per k in float32 (32x32x2 in 64 cycles) and 64 in float64
// (four 16x16x4 of 64 cycles per 4 k); the blocks a CU gets run q = ceil(blocks /
// CUs) rounds of that. Constants fitted to a sweep of 35 shapes from [64, 768] x
// [768, 3072] to [2495, 768] x [768, 3072], all layouts, aligned and not, both
// types (2.2 GHz): a launch costs about 4 us before its first MFMA (3.5 us for the
// small-product kernel, which waits for no barrier), one block alone on a CU
// reaches 0.82 (128) or 0.75 (64) of its waves' MFMA rate, several 0.97 to 1 or 0.88,
// and the small-product kernel 0.45 (float64 0.55): it re-reads its operands for
// every 32 x 32 tile through the L1. A split adds a launch and its partials'
// traffic (about 6 TB/s from the last-level cache); where the next pass takes the
// partials (`fused`: as LayerNorm or the row dots do), only the
// partials beyond the output itself. Measured, 128 -> chosen:
// [512, 384] x [384, 384] 29 -> 7 us (small-product), [1000, 256] x [256, 768]
// float64 44.6 -> 14 us (small-product), [1500, 384] x [384, 1000] 34 -> 18 us (64),
// [2495, 768] x [768, 768] 41 -> 33 us (64), [1001, 515] x [515, 1030] 36 -> 24 us.
// It does not know the epilogue, nor how long one wave's chain is: over 1473 other
// calls the geometric mean of chosen / 128 is 0.57, and the worst [2495, 1536] x
// [1536, 384] with a LayerNorm after it, 44 -> 48 us (one 64 x 64 block per CU).
static double tile_cost(int64_t M, int64_t N, int64_t K, int64_t batch, int64_t cus, int bm, int bn, int splits,
                        size_t es, bool fused) {
  const double k = (double)cdiv(cdiv(K, splits), 64 / (int64_t)es) * (64.0 / (double)es);
  const double q = (double)cdiv(cdiv(M, bm) * cdiv(N, bn) * batch * splits, cus);
  const double eff = bm == 64 ? (q > 1 ? 0.88 : 0.75) : q > 2 ? 0.97 : q > 1 ? 1.0 : 0.82;
  const double per_k = (es == 4 ? 32.0 : 64.0) * (bm / 32) * (bn / 32) / 4.0;  // four waves
  double c = 8800.0 + q * k * per_k / eff;
  const double bytes = (double)(M * N * batch) * (double)es;
  if (splits > 1) c += fused ? bytes * splits / 2700.0 : 6600.0 + bytes * (splits + 1) / 2700.0;
  return c;
}

// k per split: whole k-tiles
template <typename T>
static int64_t k_of_splits(int64_t K, int splits) {
  const int64_t kps = cdiv(cdiv(K, splits), kBKT<T>) * kBKT<T>;
  return kps < kBKT<T> ? kBKT<T> : kps;
}

// GemmArgs::fold_groups of an unsplit or thinly split range: every 192 k (a
// group is the 64 x 64 tile's 6 stages). The 128-wide plan would have split k
// over several blocks; at every 480 k the weight gradients of a block at 16 x
// 114 x 576 were further from float64 than with that plan (5.5e-7, 4.6e-7), at
// 192 they are nearer (3.9e-7), in the same time.
template <typename T>
constexpr int kFoldGroups = sizeof(T) == 4 ? 2 : 4;

// The small-product kernel with kps of k per wave: its loads' rate, or the chain
// of one wave's MFMAs (which start behind its first loads).
static double direct_cost(int64_t tiles, int64_t K, int64_t kps, int64_t cus, size_t es) {
  const double q = (double)cdiv(tiles, cus);
  const double rate = q * (double)K * (es == 4 ? 8.0 / 0.45 : 16.0 / 0.55);
  const double chain = 3500.0 + 1.35 * (es == 4 ? 32.0 : 64.0) * (double)kps;
  return 7700.0 + (rate > chain ? rate : chain);
}

// k per wave of the small-product kernel when the order of the sum is free:
// enough waves for 16 per CU, each with at least one batch of k.
template <typename T>
static int64_t direct_kps(int64_t tiles, int64_t K, int64_t cus) {
  int64_t w = 4;
  while (w < kDirectMaxWaves<T> && tiles * w < 16 * cus) w *= 2;
  return cdiv(cdiv(K, kDirectBatch<T>), w) * kDirectBatch<T>;
}

template <typename T>
static int gemm_impl(int akc, int bkc, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, int64_t sA,
                     const void* B, int64_t ldb, int64_t sB, void* C, int64_t ldc, int64_t sC, int64_t batch,
                     const void* bias, int accumulate, int force_splits, const EpiArgs& ep) {
  constexpr int VEC = MF<T>::VEC;
  GemmArgs a{};
  a.A = A;
  a.B = B;
  a.C = C;
  a.bias = bias;
  a.M = M;
  a.N = N;
  a.K = K;
  a.lda = lda;
  a.ldb = ldb;
  a.ldc = ldc;
  a.sA = sA;
  a.sB = sB;
  a.sC = sC;
  a.accumulate = accumulate;
  a.addend = ep.addend;
  a.epi = ep.epi;
  a.aux = ep.aux;
  a.colsum = ep.colsum;
  a.colsum_accumulate = ep.colsum_accumulate;
  const int64_t cus = num_cus() > 0 ? num_cus() : 256;
  const bool veca = aligned(A, 16) && lda % VEC == 0 && (batch == 1 || sA % VEC == 0) && (akc ? K % VEC == 0 : M % VEC == 0);
  const bool vecb = aligned(B, 16) && ldb % VEC == 0 && (batch == 1 || sB % VEC == 0) && (bkc ? K % VEC == 0 : N % VEC == 0);
  // The direct-to-LDS kernel addresses a tile with 32-bit byte offsets from
  // its origin: leading dimensions below 2^24 bytes keep them in range.
  constexpr int64_t kDmaMaxLd = (1 << 24) / (int64_t)sizeof(T);
  const bool dma = lda < kDmaMaxLd && ldb < kDmaMaxLd;
  // split-bf16 products: aligned float32 operands (its column sums need an
  // n-contiguous B)
  const bool x6 = std::is_same<T, float>::value && veca && vecb && g_gemm_math == DTMI_GEMM_MATH_BF16X6 &&
                  !(a.colsum && bkc) && lda < (1 << 22) && ldb < (1 << 22);
  int bm = 128, bn = 128;
  if (std::is_same<T, float>::value && dma && !x6) pick_tile(M, N, K, batch, cus, bm, bn);
  const int64_t tmn = cdiv(M, bm) * cdiv(N, bn);
  int splits = force_splits > 0 ? force_splits : choose_splits(tmn, batch, K, cus);
  bool direct = false;  // the small-product kernel
  int64_t kps = k_of_splits<T>(K, splits);
  if (dma && !x6 && force_splits <= 0 && K > 0) {
    // 7 % below the 128-wide plan's estimate before leaving it
    // the shape alone decides, so that a product gives the same bits whether or
    // not the next pass takes its partials: from one 128-wide tile per CU on,
    // the other kernels have to beat that plan with its partials taken
    const bool fused = tmn * batch >= cus;
    double best = 0.93 * tile_cost(M, N, K, batch, cus, bm, bn, splits, sizeof(T), fused);
    const int64_t t32 = cdiv(M, 32) * cdiv(N, 32) * batch;
    // Float32 products with a dimension of at most 256 keep the 128-wide plan's
    // split of k, and so the bits they had with it, whichever kernel runs. Another
    // order of the sum is no worse a rounding (all other sizes take the fastest);
    // what is kept is the trajectory of a small model's training run (dtrain's --dim
    // 128 and 256): an optimizer's first steps divide gradients by their own size,
    // and the second step's gradients of a 4-layer model of width 128 differed by
    // 3e-6. The price, also for products that train nothing: [512, 512] x [512, 128]
    // runs as 2 waves of 256 k, 9.9 us (6.0 split over 16, 23.7 on 128-wide tiles),
    // [200, 384] x [384, 384] as one chain, 12 us (29; [512, 384] x [384, 384] 7).
    const bool keep = std::is_same<T, float>::value && (M <= 256 || N <= 256 || K <= 256);
    int64_t dk = kps;
    if (keep) {
      const double c = tile_cost(M, N, K, batch, cus, 64, 64, splits, sizeof(T), fused);
      if (c < best) {
        best = c;
        bm = bn = 64;
      }
    } else {
      for (int sp = 1; sp <= 16 && (sp == 1 || K / sp >= 128); ++sp) {
        const double c = tile_cost(M, N, K, batch, cus, 64, 64, sp, sizeof(T), fused);
        if (c < best) {
          best = c;
          bm = bn = 64;
          splits = sp;
          kps = k_of_splits<T>(K, splits);
          a.fold_groups = kFoldGroups<T>;
        }
      }
      dk = direct_kps<T>(t32, K, cus);
    }
    if (cdiv(K, dk) <= kDirectMaxWaves<T> && direct_cost(t32, K, dk, cus, sizeof(T)) < best) {
      direct = true;
      splits = 1;
      kps = dk;
    }
  }
  a.tiles_m = (int)cdiv(M, bm);
  a.tiles_n = (int)cdiv(N, bn);
  const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
  DTMI_CHECK(tiles < (1LL << 31) && batch < 65536, "dtmi_gemm: problem too large");
  if (!direct) splits = (int)cdiv(K > 0 ? K : 1, kps);
  a.k_per_split = kps;
  const size_t es = sizeof(T);
  void* ws = nullptr;
  // the partials handed to the consumer (see EpiArgs::parts_out)
  const bool to_parts = ep.parts_out && splits > 1 && splits <= ep.parts_max && batch == 1 && !bias &&
                        !a.accumulate && a.epi == kEpiNone && !a.addend && !a.colsum && ldc == N;
  if (ep.parts_n) *ep.parts_n = to_parts ? splits : 1;
  if (to_parts) {
    a.ws = ep.parts_out;
  } else if (splits > 1) {
    const size_t main_bytes = (size_t)splits * batch * M * N * es;
    const size_t cs_bytes = a.colsum ? (size_t)splits * N * es : 0;
    int rc = pool_alloc(&ws, main_bytes + cs_bytes);
    if (rc) return rc;
    a.ws = ws;
    if (a.colsum) a.colsum_ws = (char*)ws + main_bytes;
  }
  // A LayerNorm of the output rows is fused into the split-K sum when the
  // rows fit the row kernel; otherwise it runs as its own pass afterwards.
  constexpr int LVW = 16 / sizeof(T);
  const int ln_nv = ep.ln_out ? ln_pick_nv(cdiv(N, 64LL * LVW)) : -1;
  const bool ln_fused = splits > 1 && ep.ln_out && batch == 1 && !a.accumulate && a.epi == kEpiNone &&
                        N % LVW == 0 && ldc == N && ln_nv > 0 && aligned(C, 16) && (!bias || aligned(bias, 16)) &&
                        (!a.addend || aligned(a.addend, 16)) && aligned(ep.ln_out, 16) && aligned(ep.ln_w, 16) &&
                        aligned(ep.ln_b, 16);
  // row dots of C with X fused into the split-K sum when C is a plain sum,
  // else a pass over the finished C
  const bool rowdot_fused = ep.rowdot_out && splits > 1 && batch == 1 && !bias && !a.addend && !a.accumulate &&
                            a.epi == kEpiNone && ldc == N && N % 64 == 0 && aligned(C, 16) &&
                            aligned(ep.rowdot_x, 16);
  bool rowdot_done = false;
  dim3 grid((unsigned)tiles, (unsigned)splits, (unsigned)batch);
  {
    TimedLaunch tl(DTMI_FAM_GEMM, 2.0 * (double)M * N * K * batch);
    if (direct) {
      launch_gemm_direct<T>(a, batch, akc, bkc);
    } else if (bm == 64) {
      launch_layout<T, 64, 64>(a, grid, akc, bkc, veca, vecb, dma);
    } else if constexpr (std::is_same<T, float>::value) {
      if (x6)
        launch_x6(a, grid, akc, bkc);
      else if (bm == 256)
        launch_layout<T, 256, 128>(a, grid, akc, bkc, veca, vecb, dma);
      else
        launch_layout<T, 128, 128>(a, grid, akc, bkc, veca, vecb, dma);
    } else {
      launch_layout<T, 128, 128>(a, grid, akc, bkc, veca, vecb, dma);
    }
    if (splits > 1 && !ln_fused && !to_parts) {
      int64_t total = batch * M * N;
      int rg = (int)(cdiv(total, 256 * 4) < 8192 ? cdiv(total, 256 * 4) : 8192);
      GemmArgs r = a;
      r.ws = nullptr;
      const bool plain = a.addend == nullptr && a.epi == kEpiNone && !a.accumulate;
      constexpr int V = 16 / sizeof(T);
      const bool vec_ok = N % V == 0 && ldc % V == 0 && (batch == 1 || sC % V == 0) && aligned(C, 16) &&
                          (!bias || aligned(bias, 16)) && (!a.addend || aligned(a.addend, 16)) &&
                          (!a.aux || aligned(a.aux, 16));
      if constexpr (std::is_same<T, float>::value) {
        if (rowdot_fused) {
          splitk_rowdot_kernel<<<rg, 256, 0, stream()>>>(r, (const float*)ws, splits, (const float*)ep.rowdot_x,
                                                          (float*)ep.rowdot_out, ep.rowdot_T);
          rowdot_done = true;
        }
      }
      if (rowdot_done) {
      } else if (plain && vec_ok)
        splitk_reduce_kernel<T, true, V><<<rg, 256, 0, stream()>>>(r, (const T*)ws, splits, batch);
      else if (vec_ok)
        splitk_reduce_kernel<T, false, V><<<rg, 256, 0, stream()>>>(r, (const T*)ws, splits, batch);
      else if (plain)
        splitk_reduce_kernel<T, true, 1><<<rg, 256, 0, stream()>>>(r, (const T*)ws, splits, batch);
      else
        splitk_reduce_kernel<T, false, 1><<<rg, 256, 0, stream()>>>(r, (const T*)ws, splits, batch);
    }
  }
  if (ln_fused) {
    // split-K partials, bias and residual in; C and the LayerNorm out
    TimedLaunch tl(DTMI_FAM_OTHER, (double)M * N * sizeof(T) * (splits + (a.addend ? 3 : 2)));
    GemmArgs r = a;
    r.ws = nullptr;
    const unsigned lg = (unsigned)cdiv(M, 4);
#define CALL_LN_S(NV, S2)                                                                                      \
  splitk_ln_kernel<T, NV, LVW, S2><<<lg, 256, 0, stream()>>>(r, (const T*)ws, splits, (T*)ep.ln_out,               \
                                                              (T*)ep.ln_mean, (T*)ep.ln_rstd, (const T*)ep.ln_w, \
                                                              (const T*)ep.ln_b, (T)ep.ln_eps)
#define CALL_LN(NV)          \
  if (splits == 2)           \
    CALL_LN_S(NV, true);     \
  else                       \
    CALL_LN_S(NV, false)
    LN_NV_SWITCH(ln_nv, CALL_LN)
#undef CALL_LN
#undef CALL_LN_S
  }
  if constexpr (std::is_same<T, float>::value) {
    if (ep.rowdot_out && !rowdot_done) {
      TimedLaunch tl(DTMI_FAM_OTHER, 2.0 * (double)M * N * sizeof(T));
      const int64_t nv = M * N / 4;
      rowdot64_kernel<<<(unsigned)(cdiv(nv, 256) < 8192 ? cdiv(nv, 256) : 8192), 256, 0, stream()>>>(
          (const float*)C, (const float*)ep.rowdot_x, (float*)ep.rowdot_out, M, N, ep.rowdot_T);
    }
  }
  hipError_t le = hipGetLastError();
  if (ws) pool_free(ws);
  if (le != hipSuccess) return fail_hip(le, "gemm kernels", __FILE__, __LINE__);
  if (ep.ln_out && !ln_fused)  // the LayerNorm as its own pass over C
    return dtmi_layernorm_fwd(std::is_same<T, float>::value ? DTMI_F32 : DTMI_F64, ep.ln_out, ep.ln_mean, ep.ln_rstd,
                              C, ep.ln_w, ep.ln_b, M, N, ep.ln_eps);
  return DTMI_OK;
}

static int gemm_dispatch(int dtype, int akc, int bkc, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda,
                         int64_t sA, const void* B, int64_t ldb, int64_t sB, void* C, int64_t ldc, int64_t sC,
                         int64_t batch, const void* bias, int accumulate, int force_splits,
                         const EpiArgs& ep = EpiArgs()) {
  DTMI_DTYPE_OK(dtype);
  DTMI_CHECK(M >= 0 && N >= 0 && K >= 0 && batch >= 1, "dtmi_gemm: bad sizes M=%lld N=%lld K=%lld batch=%lld",
             (long long)M, (long long)N, (long long)K, (long long)batch);
  if (M == 0 || N == 0) return DTMI_OK;
  DTMI_CHECK(C != nullptr && (K == 0 || (A && B)), "dtmi_gemm: NULL pointer");
  DTMI_CHECK(ldc >= N, "dtmi_gemm: ldc %lld < N %lld", (long long)ldc, (long long)N);
  DTMI_CHECK(K == 0 || (akc ? lda >= K : lda >= M), "dtmi_gemm: lda too small");
  DTMI_CHECK(K == 0 || (bkc ? ldb >= K : ldb >= N), "dtmi_gemm: ldb too small");
  DTMI_CHECK(ep.epi == kEpiNone || ep.aux != nullptr, "dtmi_gemm: GELU epilogue without its array");
  DTMI_CHECK(ep.colsum == nullptr || batch == 1, "dtmi_gemm: column sums are for unbatched products");
  if (dtype == DTMI_F32)
    return gemm_impl<float>(akc, bkc, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, batch, bias, accumulate,
                            force_splits, ep);
  return gemm_impl<double>(akc, bkc, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, batch, bias, accumulate,
                           force_splits, ep);
}

}  // namespace dtmi

using namespace dtmi;

DTMI_EXPORT int dtmi_set_gemm_math(int math) {
  DTMI_BODY_BEGIN
  DTMI_CHECK(math == DTMI_GEMM_MATH_F32 || math == DTMI_GEMM_MATH_BF16X6, "dtmi_set_gemm_math: unknown mode %d",
             math);
  g_gemm_math = math;
  return DTMI_OK;
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_get_gemm_math(int* math) {
  DTMI_BODY_BEGIN
  DTMI_CHECK(math != nullptr, "dtmi_get_gemm_math: NULL pointer");
  *math = g_gemm_math;
  return DTMI_OK;
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_gemm(int dtype, int a_kcontig, int b_kcontig, int64_t M, int64_t N, int64_t K, const void* A,
                          int64_t lda, int64_t strideA, const void* B, int64_t ldb, int64_t strideB, void* C,
                          int64_t ldc, int64_t strideC, int64_t batch, const void* bias, int accumulate,
                          int splits) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  return gemm_dispatch(dtype, a_kcontig ? 1 : 0, b_kcontig ? 1 : 0, M, N, K, A, lda, strideA, B, ldb, strideB, C, ldc,
                       strideC, batch, bias, accumulate, splits);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_fwd(int dtype, void* Y, const void* X, const void* W, const void* b, int64_t M,
                                int64_t K, int64_t N) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  return gemm_dispatch(dtype, 1, 0, M, N, K, X, K, 0, W, N, 0, Y, N, 0, 1, b, 0, 0);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_fwd_fused(int dtype, void* Y, void* act, const void* X, const void* W, const void* b,
                                      const void* residual, int64_t M, int64_t K, int64_t N) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  EpiArgs ep;
  ep.addend = residual;
  ep.epi = act ? kEpiGeluFwd : kEpiNone;
  ep.aux = act;
  DTMI_CHECK(!(act && residual), "dtmi_linear_fwd_fused: GELU and residual are not fused together");
  return gemm_dispatch(dtype, 1, 0, M, N, K, X, K, 0, W, N, 0, Y, N, 0, 1, b, 0, 0, ep);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_fwd_ln(int dtype, void* Y, void* H, void* mean, void* rstd, const void* X, const void* W,
                                   const void* b, const void* residual, const void* ln_w, const void* ln_b, double eps,
                                   int64_t M, int64_t K, int64_t N) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  DTMI_CHECK(H && mean && rstd && ln_w && ln_b, "dtmi_linear_fwd_ln: NULL LayerNorm pointer");
  DTMI_CHECK(H != Y, "dtmi_linear_fwd_ln: the LayerNorm output must not be Y");
  EpiArgs ep;
  ep.addend = residual;
  ep.ln_out = H;
  ep.ln_mean = mean;
  ep.ln_rstd = rstd;
  ep.ln_w = ln_w;
  ep.ln_b = ln_b;
  ep.ln_eps = eps;
  return gemm_dispatch(dtype, 1, 0, M, N, K, X, K, 0, W, N, 0, Y, N, 0, 1, b, 0, 0, ep);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_bwd_dx_gelu(int dtype, void* dX, const void* dY, const void* W, const void* pre,
                                        int64_t M, int64_t K, int64_t N) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  DTMI_CHECK(pre != nullptr, "dtmi_linear_bwd_dx_gelu: NULL pre-activation");
  EpiArgs ep;
  ep.epi = kEpiGeluBwd;
  ep.aux = const_cast<void*>(pre);
  return gemm_dispatch(dtype, 1, 1, M, K, N, dY, N, 0, W, N, 0, dX, K, 0, 1, nullptr, 0, 0, ep);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_bwd_dx(int dtype, void* dX, const void* dY, const void* W, int64_t M, int64_t K,
                                   int64_t N, int accumulate) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  // dX[m, k] = sum_n dY[m, n] W[k, n]: A = dY (k-contiguous over n), B(n, k) = W[k, n] (k-contiguous)
  return gemm_dispatch(dtype, 1, 1, M, K, N, dY, N, 0, W, N, 0, dX, K, 0, 1, nullptr, accumulate, 0);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_bwd_dx_parts(int dtype, void* parts, int max_parts, int* nparts, const void* dY,
                                         const void* W, int64_t M, int64_t K, int64_t N) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  DTMI_CHECK(parts && nparts && max_parts >= 1, "dtmi_linear_bwd_dx_parts: NULL parts / nparts or max_parts < 1");
  EpiArgs ep;
  ep.parts_out = parts;
  ep.parts_max = max_parts;
  ep.parts_n = nparts;
  *nparts = 1;
  return gemm_dispatch(dtype, 1, 1, M, K, N, dY, N, 0, W, N, 0, parts, K, 0, 1, nullptr, 0, 0, ep);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_bwd_dx_rowdot(int dtype, void* dX, const void* dY, const void* W, const void* X,
                                          void* rowdot, int64_t M, int64_t K, int64_t N, int64_t T) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  DTMI_CHECK(dtype == DTMI_F32, "dtmi_linear_bwd_dx_rowdot: float32 only");
  DTMI_CHECK(M >= 0 && K > 0 && N >= 0 && T > 0 && K % 64 == 0 && M % T == 0,
             "dtmi_linear_bwd_dx_rowdot: needs K %% 64 == 0 and M %% T == 0 (M=%lld K=%lld T=%lld)", (long long)M,
             (long long)K, (long long)T);
  DTMI_CHECK(X && rowdot && aligned(dX, 16) && aligned(X, 16), "dtmi_linear_bwd_dx_rowdot: NULL or unaligned X / dX");
  EpiArgs ep;
  ep.rowdot_x = X;
  ep.rowdot_out = rowdot;
  ep.rowdot_T = T;
  return gemm_dispatch(dtype, 1, 1, M, K, N, dY, N, 0, W, N, 0, dX, K, 0, 1, nullptr, 0, 0, ep);
  DTMI_BODY_END
}

DTMI_EXPORT int dtmi_linear_bwd_dw(int dtype, void* dW, void* db, const void* X, const void* dY, int64_t M,
                                   int64_t K, int64_t N, int accumulate) {
  DTMI_BODY_BEGIN
  DTMI_REQUIRE_INIT();
  // dW[k, n] = sum_m X[m, k] dY[m, n]: A(k, m) = X[m, k] (k-major storage), B(m, n) = dY[m, n];
  // db[n] = sum_m dY[m, n], the column sums of B, taken inside the same GEMM
  if (K == 0) return db ? dtmi_colsum(dtype, db, dY, M, N, accumulate) : DTMI_OK;  // no dW tiles to carry db
  EpiArgs ep;
  ep.colsum = db;
  ep.colsum_accumulate = accumulate;
  return gemm_dispatch(dtype, 0, 0, K, N, M, X, K, 0, dY, N, 0, dW, N, 0, 1, nullptr, accumulate, 0, ep);
  DTMI_BODY_END
}
