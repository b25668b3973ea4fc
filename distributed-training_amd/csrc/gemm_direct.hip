// Small products: C = sum_k A(m,k) B(k,n) with the k range split over the waves
// of a block and the operands read straight into MFMA fragments.
//
// What bounds a small product is not the matrix cores' rate but how few of
// them it reaches: [512, 512] x [512, 128] is four 128 x 128 tiles, four blocks
// on 256 CUs, and each of their waves runs K / 2 MFMAs of 64 cycles per 32 x 32
// piece one after the other. Here a block owns one 32 x 32 tile, its nw waves
// take consecutive ranges of k, and their partial tiles are added through LDS in
// wave order: the four tiles become 64 blocks, of up to 16 waves where the order
// of the sum is free (the dispatch says where), with no second launch to sum
// partials. The waves share no operand data (each has its own k), so nothing is
// staged in LDS and there is no barrier before the sum; each wave keeps one batch
// of k in flight in registers while it multiplies the one before.
//
// Loads: a k-contiguous operand gives a lane its VEC k-values of a row as one
// 16-byte vector, an m/n-contiguous one a k-row's 32 (16) neighbours as 4-byte
// (8-byte) elements. Neither needs more than element alignment (global vector
// loads take any 4-byte address), so odd leading dimensions run at full width.
// Rows and columns past the edge are clamped onto the last one (they feed only
// outputs that are not stored); a wave's last, partial batch is read element by
// element, clamped and zeroed at k >= the range's end.
#include <type_traits>

#include "common.h"
#include "gemm_common.h"
#include "gemm_direct.h"

namespace dtmi {

// 16-byte vector at an element-aligned address
template <typename T>
struct UVec;
template <>
struct UVec<float> {
  typedef MF<float>::vec_t __attribute__((aligned(4))) type;
};
template <>
struct UVec<double> {
  typedef MF<double>::vec_t __attribute__((aligned(8))) type;
};

// One operand's share of a wave: R MFMA tiles of MT rows (columns) along m/n by
// KB of k per batch.
template <typename T, bool KCONTIG, int R, int KB>
struct DirectSrc {
  static constexpr int MT = MF<T>::MT, VEC = MF<T>::VEC, NCH = KB / 8;
  typedef typename MF<T>::vec_t VT;
  const char* base;  // wave-uniform: the current batch's first k
  unsigned off[R];   // this lane's byte offset from it
  int64_t ldb;       // bytes between k-rows (m/n-contiguous)

  __device__ __forceinline__ void init(const T* __restrict__ P, int64_t ld, int64_t mn0, int64_t MN, int64_t k0, int g,
                                       int c) {
    base = reinterpret_cast<const char*>(KCONTIG ? P + mn0 * ld + k0 : P + k0 * ld + mn0);
    ldb = ld * (int64_t)sizeof(T);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      int64_t r = mn0 + i * MT + c;
      r = (r < MN ? r : MN - 1) - mn0;
      off[i] = (unsigned)((KCONTIG ? r * ld + VEC * g : (int64_t)VEC * g * ld + r) * (int64_t)sizeof(T));
    }
  }
  __device__ __forceinline__ void load(VT (&v)[R][NCH]) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch) {
        if constexpr (KCONTIG) {
          v[i][ch] = *reinterpret_cast<const typename UVec<T>::type*>(base + off[i] + 8 * ch * sizeof(T));
        } else {
#pragma unroll
          for (int s = 0; s < VEC; ++s) v[i][ch][s] = *reinterpret_cast<const T*>(base + (8 * ch + s) * ldb + off[i]);
        }
      }
    base += KCONTIG ? (int64_t)KB * (int64_t)sizeof(T) : (int64_t)KB * ldb;
  }
  // the last `left` (< KB) values of k: element loads clamped to k = left - 1,
  // zeros from `left` on
  __device__ __forceinline__ void load_tail(VT (&v)[R][NCH], int left, int g) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch)
#pragma unroll
        for (int s = 0; s < VEC; ++s) {
          const int k = 8 * ch + VEC * g + s;
          const int64_t kc = (k < left ? k : left - 1) - VEC * g;  // relative to this lane's offset
          const T x = *reinterpret_cast<const T*>(base + (int64_t)off[i] + kc * (KCONTIG ? (int64_t)sizeof(T) : ldb));
          v[i][ch][s] = k < left ? x : T(0);
        }
  }
};

template <typename T>
struct DirectTile {
  static constexpr int EDGE = 32;                      // block tile
  static constexpr int R = EDGE / MF<T>::MT;           // MFMA tiles per edge
  static constexpr int REGS = R * R * MF<T>::NACC;     // accumulators per lane
  static constexpr int KB = kDirectBatch<T>;
};

template <typename T, bool AKC, bool BKC>
__global__ void __launch_bounds__(64 * kDirectMaxWaves<T>) gemm_direct_kernel(GemmArgs a) {
  using MFT = MF<T>;
  using D = DirectTile<T>;
  constexpr int MT = MFT::MT, NACC = MFT::NACC, VEC = MFT::VEC, R = D::R, KB = D::KB, NCH = KB / 8;
  constexpr int CPT = kBKT<T> / 8;  // 8-wide chunks per k-tile of the tiled kernels
  typedef typename MFT::vec_t VT;
  extern __shared__ __attribute__((aligned(16))) char lds_raw[];

  int tm, tn;
  tile_coords(a, tm, tn);
  const int64_t m0 = (int64_t)tm * D::EDGE, n0 = (int64_t)tn * D::EDGE;
  const int64_t batch = blockIdx.z;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = (int)(blockDim.x >> 6);
  const int g = lane / MT, c = lane % MT;
  // this wave's k range (the host gives every wave at least one k)
  const int64_t kbeg = (int64_t)wave * a.k_per_split;
  const int64_t kend = kbeg + a.k_per_split < a.K ? kbeg + a.k_per_split : a.K;
  const int kn = kend > kbeg ? (int)(kend - kbeg) : 0;

  typename MFT::acc_t acc[R][R];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < R; ++j) acc[i][j] = typename MFT::acc_t(0);
  const bool take_colsum = a.colsum != nullptr && tm == 0;
  double cs[R];
#pragma unroll
  for (int j = 0; j < R; ++j) cs[j] = 0.0;

  DirectSrc<T, AKC, R, KB> sa;
  DirectSrc<T, BKC, R, KB> sb;
  sa.init((const T*)a.A + batch * a.sA, a.lda, m0, a.M, kbeg, g, c);
  sb.init((const T*)a.B + batch * a.sB, a.ldb, n0, a.N, kbeg, g, c);
  auto mul = [&](const VT (&x)[R][NCH], const VT (&y)[R][NCH], int chunks) {
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      if (ch >= chunks) break;
#pragma unroll
      for (int s = 0; s < VEC; ++s)
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j) acc[i][j] = MFT::mma(x[i][ch][s], y[j][ch][s], acc[i][j]);
    }
    if (take_colsum) {
      // every 16 k: the sum in k order, then into the running float64 sum, as
      // the tiled kernels take it (k past the range is zero). A lane group
      // holds VEC of each G * VEC consecutive k; the others' come by shuffle.
#pragma unroll
      for (int j = 0; j < R; ++j)
#pragma unroll
        for (int c0 = 0; c0 < NCH; c0 += CPT) {
          T t = T(0);
#pragma unroll
          for (int ch = c0; ch < c0 + CPT; ++ch)
#pragma unroll
            for (int gg = 0; gg < MFT::G; ++gg)
#pragma unroll
              for (int s = 0; s < VEC; ++s) t = t + __shfl(y[j][ch][s], gg * MT + c, 64);
          cs[j] += (double)t;
        }
    }
  };
  const int nb = kn / KB, left = kn - nb * KB;
  VT x0[R][NCH], y0[R][NCH], x1[R][NCH], y1[R][NCH];
  if (nb > 0) {
    sa.load(x0);
    sb.load(y0);
    int b = 0;
    for (; b + 2 <= nb; b += 2) {
      sa.load(x1);
      sb.load(y1);
      mul(x0, y0, NCH);
      if (b + 2 < nb) {
        sa.load(x0);
        sb.load(y0);
      }
      mul(x1, y1, NCH);
    }
    if (b < nb) mul(x0, y0, NCH);
  }
  if (left > 0) {
    sa.load_tail(x0, left, g);
    sb.load_tail(y0, left, g);
    mul(x0, y0, (left + 7) / 8);
  }

  T* C = (T*)a.C + batch * a.sC;
  if (nw == 1) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j)
#pragma unroll
        for (int r = 0; r < NACC; ++r) {
          const int64_t m = m0 + i * MT + MFT::row(r, g), n = n0 + j * MT + c;
          if (m < a.M && n < a.N) epilogue_store<T>(a, C, a.ldc, m, n, acc[i][j][r], batch);
        }
  } else {
    // partial tiles [wave][register][lane]; wave w then sums registers w, w + nw,
    // ... over the waves in order
    T* part = reinterpret_cast<T*>(lds_raw);
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j)
#pragma unroll
        for (int r = 0; r < NACC; ++r) part[(wave * D::REGS + (i * R + j) * NACC + r) * 64 + lane] = acc[i][j][r];
    __syncthreads();
    for (int q = wave; q < D::REGS; q += nw) {
      T v = part[q * 64 + lane];
      for (int w = 1; w < nw; ++w) v = v + part[(w * D::REGS + q) * 64 + lane];
      const int t = q / NACC, r = q % NACC;
      const int64_t m = m0 + (t / R) * MT + MFT::row(r, g), n = n0 + (t % R) * MT + c;
      if (m < a.M && n < a.N) epilogue_store<T>(a, C, a.ldc, m, n, v, batch);
    }
  }
  if (take_colsum) {  // block-uniform
    // the waves' sums in order, each rounded to T as a split's is
    double* red = reinterpret_cast<double*>(lds_raw);
    if (nw > 1) __syncthreads();  // the partial tiles are read
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (g == 0) red[wave * D::EDGE + j * MT + c] = cs[j];
    __syncthreads();
    for (int n = threadIdx.x; n < D::EDGE; n += blockDim.x) {
      T v = (T)red[n];
      for (int w = 1; w < nw; ++w) v = v + (T)red[w * D::EDGE + n];
      finish_colsum<T>(a, (double)v, n0 + n, 0);
    }
  }
}

template <typename T>
void launch_gemm_direct(GemmArgs a, int64_t batch, int akc, int bkc) {
  using D = DirectTile<T>;
  a.tiles_m = (int)cdiv(a.M, D::EDGE);
  a.tiles_n = (int)cdiv(a.N, D::EDGE);
  a.ws = nullptr;
  a.colsum_ws = nullptr;
  const int nw = (int)cdiv(a.K, a.k_per_split);  // every wave gets some k; the plan keeps their limit
  size_t lds = nw > 1 ? (size_t)nw * D::REGS * 64 * sizeof(T) : 0;
  if (a.colsum) {
    const size_t cb = (size_t)nw * D::EDGE * sizeof(double);
    lds = lds > cb ? lds : cb;
  }
  const dim3 grid((unsigned)(a.tiles_m * a.tiles_n), 1, (unsigned)batch);
  const unsigned th = 64u * (unsigned)nw;
  if (akc && bkc)
    gemm_direct_kernel<T, true, true><<<grid, th, lds, stream()>>>(a);
  else if (akc)
    gemm_direct_kernel<T, true, false><<<grid, th, lds, stream()>>>(a);
  else if (bkc)
    gemm_direct_kernel<T, false, true><<<grid, th, lds, stream()>>>(a);
  else
    gemm_direct_kernel<T, false, false><<<grid, th, lds, stream()>>>(a);
}

template void launch_gemm_direct<float>(GemmArgs, int64_t, int, int);
template void launch_gemm_direct<double>(GemmArgs, int64_t, int, int);

}  // namespace dtmi
