// The float32 / float64 MFMA GEMM kernels (block tiles staged in LDS) and their
// launches; gemm.hip holds the layout notes and the dispatch. One translation
// unit per tile and type instantiates launch_layout.
#pragma once

#include <type_traits>
#include <utility>

#include "bufrsrc.h"
#include "common.h"
#include "gelu.h"
#include "gemm_common.h"

namespace dtmi {

constexpr int kKC = 8;

// One operand tile of BMN rows/columns (along M or N) by kBK.
template <typename T, bool KCONTIG, int BMN>
struct TileLayout {
  static constexpr int VEC = MF<T>::VEC;
  static constexpr int kBK = kBKT<T>;
  // k-contiguous: [mn][kBK + VEC]; mn-contiguous: [kBK][BMN + 8]
  static constexpr int STRIDE = KCONTIG ? (kBK + VEC) : (BMN + 8);
  static constexpr int SIZE = KCONTIG ? BMN * STRIDE : kBK * STRIDE;
  static constexpr int NVEC = BMN * kBK / VEC / 256;  // 16-byte vectors per thread per tile
};

template <typename T, bool KCONTIG, int BMN>
struct TileRegs {
  typename MF<T>::vec_t v[TileLayout<T, KCONTIG, BMN>::NVEC];
};

// Global -> registers for one BMN x kBK operand tile (mn0 = first row/col of
// the tile along M or N, k0 = first k), element by element: any alignment,
// out-of-range elements read as 0.
template <typename T, bool KCONTIG, int BMN>
__device__ __forceinline__ void load_tile(TileRegs<T, KCONTIG, BMN>& r, const T* __restrict__ P, int64_t ld,
                                          int64_t mn0, int64_t MN, int64_t k0, int64_t kend) {
  using L = TileLayout<T, KCONTIG, BMN>;
  constexpr int VEC = L::VEC;
  constexpr int kBK = L::kBK;
#pragma unroll
  for (int i = 0; i < L::NVEC; ++i) {
    const int f = threadIdx.x + 256 * i;
    const int64_t mn = mn0 + (KCONTIG ? f / (kBK / VEC) : (f % (BMN / VEC)) * VEC);
    const int64_t k = k0 + (KCONTIG ? (f % (kBK / VEC)) * VEC : f / (BMN / VEC));
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const int64_t mm = KCONTIG ? mn : mn + e;
      const int64_t kk = KCONTIG ? k + e : k;
      r.v[i][e] = (mm < MN && kk < kend) ? (KCONTIG ? P[mm * ld + kk] : P[kk * ld + mm]) : T(0);
    }
  }
}

// Per-thread source pointers for the vector loads of one k-tile. Rows (or
// columns) past the matrix edge are clamped onto its last row/column: they
// feed only output rows/columns that the epilogue never stores.
template <typename T, bool KCONTIG, int BMN>
struct TilePtr {
  const T* p[TileLayout<T, KCONTIG, BMN>::NVEC];
};

template <typename T, bool KCONTIG, int BMN>
__device__ __forceinline__ void init_ptr(TilePtr<T, KCONTIG, BMN>& t, const T* __restrict__ P, int64_t ld,
                                         int64_t mn0, int64_t MN, int64_t kbeg) {
  using L = TileLayout<T, KCONTIG, BMN>;
  constexpr int VEC = L::VEC;
  constexpr int kBK = L::kBK;
#pragma unroll
  for (int i = 0; i < L::NVEC; ++i) {
    const int f = threadIdx.x + 256 * i;
    if (KCONTIG) {
      int64_t mn = mn0 + f / (kBK / VEC);
      mn = mn < MN ? mn : MN - 1;
      t.p[i] = P + mn * ld + kbeg + (f % (kBK / VEC)) * VEC;
    } else {
      int64_t mn = mn0 + (f % (BMN / VEC)) * VEC;
      mn = mn < MN ? mn : MN - VEC;
      t.p[i] = P + (kbeg + f / (BMN / VEC)) * ld + mn;
    }
  }
}

// A k-tile wholly in range; the pointers advance by `step` elements to the next.
template <typename T, bool KCONTIG, int BMN>
__device__ __forceinline__ void load_full(TileRegs<T, KCONTIG, BMN>& r, TilePtr<T, KCONTIG, BMN>& t, int64_t step) {
#pragma unroll
  for (int i = 0; i < TileLayout<T, KCONTIG, BMN>::NVEC; ++i) {
    r.v[i] = *reinterpret_cast<const typename MF<T>::vec_t*>(t.p[i]);
    t.p[i] += step;
  }
}

// The last k-tile when it extends past kend: the same number of loads as a
// full tile, from addresses clamped into [kbeg, kend) (k past kend is zeroed
// when the tile is stored to LDS, see store_tile and dma_tail_store).
template <typename T, bool KCONTIG, int BMN>
__device__ __forceinline__ void load_tail(TileRegs<T, KCONTIG, BMN>& r, const TilePtr<T, KCONTIG, BMN>& t,
                                          int64_t ld, int64_t k0, int64_t kend) {
  using L = TileLayout<T, KCONTIG, BMN>;
  constexpr int VEC = L::VEC;
  constexpr int kBK = L::kBK;
#pragma unroll
  for (int i = 0; i < L::NVEC; ++i) {
    const int f = threadIdx.x + 256 * i;
    const T* q;
    if (KCONTIG) {
      const int64_t k = k0 + (f % (kBK / VEC)) * VEC;
      q = t.p[i] - (k < kend ? 0 : k - (kend - VEC));
    } else {
      const int64_t k = k0 + f / (BMN / VEC);
      q = t.p[i] - (k < kend ? 0 : (k - (kend - 1)) * ld);
    }
    r.v[i] = *reinterpret_cast<const typename MF<T>::vec_t*>(q);
  }
}

// Registers -> LDS; TAIL: vectors whose k is `left` or more past the tile's first as zeros.
template <bool TAIL, typename T, bool KCONTIG, int BMN>
__device__ __forceinline__ void store_tile(T* __restrict__ lds, const TileRegs<T, KCONTIG, BMN>& r, int left) {
  using L = TileLayout<T, KCONTIG, BMN>;
  constexpr int VEC = L::VEC;
  constexpr int kBK = L::kBK;
#pragma unroll
  for (int i = 0; i < L::NVEC; ++i) {
    const int f = threadIdx.x + 256 * i;
    const int row = KCONTIG ? f / (kBK / VEC) : f / (BMN / VEC);
    const int col = (KCONTIG ? f % (kBK / VEC) : f % (BMN / VEC)) * VEC;
    const bool in = !TAIL || (KCONTIG ? col : row) < left;
    *reinterpret_cast<typename MF<T>::vec_t*>(lds + row * L::STRIDE + col) = in ? r.v[i] : typename MF<T>::vec_t(0);
  }
}

// The VEC k-values lane (group g, position c) feeds for operand rows/cols
// `base + c` at chunk `kk`.
template <typename T, bool KCONTIG, int BMN>
__device__ __forceinline__ typename MF<T>::vec_t read_frag(const T* __restrict__ lds, int base, int kk, int g, int c) {
  using L = TileLayout<T, KCONTIG, BMN>;
  constexpr int VEC = L::VEC;
  typename MF<T>::vec_t v;
  if (KCONTIG) {
    v = *reinterpret_cast<const typename MF<T>::vec_t*>(lds + (base + c) * L::STRIDE + kk + VEC * g);
  } else {
#pragma unroll
    for (int s = 0; s < VEC; ++s) v[s] = lds[(kk + VEC * g + s) * L::STRIDE + base + c];
  }
  return v;
}

// A wave's TM x TN MFMA accumulators (its tile starts at row m0, column n0):
// split-K partials go to the workspace as they are; otherwise the fused
// epilogue writes C (and aux).
template <typename T, int TM, int TN, bool FAST_EPI = false>
__device__ __forceinline__ void write_acc(const GemmArgs& a, const typename MF<T>::acc_t (&acc)[TM][TN], int64_t m0,
                                          int64_t n0, int g, int c, int split, int64_t batch) {
  using MFT = MF<T>;
  constexpr int MT = MFT::MT, NACC = MFT::NACC;
  const bool to_ws = a.ws != nullptr;
  T* C = to_ws ? (T*)a.ws + ((int64_t)split * gridDim.z + batch) * a.M * a.N : (T*)a.C + batch * a.sC;
  const int64_t ldc = to_ws ? a.N : a.ldc;
  if constexpr (FAST_EPI && std::is_same<T, float>::value) {
    if ((to_ws || (a.addend == nullptr && !a.accumulate)) && m0 + TM * MT <= a.M && n0 + TN * MT <= a.N) {
      // A whole wave tile in range with no residual or accumulation (every
      // split-K partial, the bias-only products, the GELU epilogues): buffer
      // accesses off the wave tile's corner -- one lane offset, and per
      // element a wave-uniform offset, so no per-element address arithmetic
      // on the SIMD the MFMAs share. The GELU backward's pre-activation of a
      // row of MFMA tiles is read before its first store (the stores may
      // alias it as far as the compiler can tell). Same operations as
      // epilogue_store.
      const int64_t corner = m0 * ldc + n0;
      const float* bias = to_ws ? nullptr : (const float*)a.bias;
      const Rsrc rc = make_rsrc(C + corner, ~0ull);
      const Rsrc rx = make_rsrc(to_ws ? C : (const float*)a.aux + batch * a.sC + corner, ~0ull);
      const uint32_t voff = (uint32_t)((4 * g * ldc + c) * 4);
      auto run = [&](auto modec) {
        constexpr int MODE = decltype(modec)::value;  // an epilogue kind
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          float x[TN][NACC];
          if constexpr (MODE == kEpiGeluBwd) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
              for (int r = 0; r < NACC; ++r)
                x[j][r] = buf_load1(rx, voff, (uint32_t)(((i * MT + MFT::row(r, 0)) * ldc + j * MT) * 4));
          }
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            const float bn = bias ? bias[n0 + j * MT + c] : 0.f;
#pragma unroll
            for (int r = 0; r < NACC; ++r) {
              const uint32_t so = (uint32_t)(((i * MT + MFT::row(r, 0)) * ldc + j * MT) * 4);
              float v = acc[i][j][r];
              if (bias) v = v + bn;
              if constexpr (MODE == kEpiGeluFwd) buf_store1(gelu_f<float>(v), rx, voff, so);
              if constexpr (MODE == kEpiGeluBwd) v = gelu_b<float>(x[j][r], v);
              buf_store1(v, rc, voff, so);
            }
          }
        }
      };
      const int epi = to_ws ? kEpiNone : a.epi;
      if (epi == kEpiGeluBwd)
        run(std::integral_constant<int, kEpiGeluBwd>());
      else if (epi == kEpiGeluFwd)
        run(std::integral_constant<int, kEpiGeluFwd>());
      else
        run(std::integral_constant<int, kEpiNone>());
      return;
    }
  }
  const bool plain = to_ws || (a.addend == nullptr && a.epi == kEpiNone && !a.accumulate);
  if (plain) {  // raw split-K partial, or v + bias
    const T* bias = to_ws ? nullptr : (const T*)a.bias;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t n = n0 + j * MT + c;
        if (n >= a.N) continue;
        const T bn = bias ? bias[n] : T(0);
#pragma unroll
        for (int r = 0; r < NACC; ++r) {
          const int64_t m = m0 + i * MT + MFT::row(r, g);
          if (m >= a.M) continue;
          T v = acc[i][j][r];
          if (bias) v = v + bn;
          C[m * ldc + n] = v;
        }
      }
  } else {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t n = n0 + j * MT + c;
        if (n >= a.N) continue;
#pragma unroll
        for (int r = 0; r < NACC; ++r) {
          const int64_t m = m0 + i * MT + MFT::row(r, g);
          if (m >= a.M) continue;
          epilogue_store<T>(a, C, ldc, m, n, acc[i][j][r], batch);
        }
      }
  }
}

// Leading dimensions beyond the 32-bit offsets of gemm_dma_kernel: registers ->
// LDS. VECA / VECB: a 16-byte granular operand is read as vectors through
// per-thread pointers advanced by a k-tile (float32 [256, 4096] x [4096, 256],
// rows of A 2^24 bytes apart: 36 us, 59 element by element); others element by
// element. Block tile BM x BN, 4 waves in a 2 x 2 grid of (BM/2) x (BN/2) wave
// tiles.
template <typename T, int BM, int BN, bool AKC, bool BKC, bool VECA, bool VECB>
__global__ void __launch_bounds__(256, 2) gemm_kernel(GemmArgs a) {
  constexpr int kBK = kBKT<T>;
  using MFT = MF<T>;
  using LA = TileLayout<T, AKC, BM>;
  using LB = TileLayout<T, BKC, BN>;
  constexpr int MT = MFT::MT, VEC = MFT::VEC, NACC = MFT::NACC;
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int TM = WM / MT, TN = WN / MT;
  constexpr int NCH = kBK / kKC;  // 8-wide k chunks per k-tile
  __shared__ __attribute__((aligned(16))) T lds[2 * (LA::SIZE + LB::SIZE)];

  int tm, tn;
  tile_coords(a, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int split = blockIdx.y;
  const int64_t batch = blockIdx.z;
  const int64_t kbeg = (int64_t)split * a.k_per_split;
  const int64_t kend = kbeg + a.k_per_split < a.K ? kbeg + a.k_per_split : a.K;
  const T* A = (const T*)a.A + batch * a.sA;
  const T* B = (const T*)a.B + batch * a.sB;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane / MT, c = lane % MT;
  const int wm0 = (wave >> 1) * WM, wn0 = (wave & 1) * WN;

  typename MFT::acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = typename MFT::acc_t(0);

  // LDS is double-buffered with one barrier per k-tile: iteration kt issues
  // the global loads of tile kt+1 into registers, computes tile kt from LDS
  // stage kt&1 while they are in flight, then stores them to the other stage.
  TileRegs<T, AKC, BM> ra;
  TileRegs<T, BKC, BN> rb;
  const int64_t ntiles = kend > kbeg ? (kend - kbeg + kBK - 1) / kBK : 0;
  const int64_t nfull = kend > kbeg ? (kend - kbeg) / kBK : 0;
  TilePtr<T, AKC, BM> pa;
  TilePtr<T, BKC, BN> pb;
  if (VECA) init_ptr<T, AKC, BM>(pa, A, a.lda, m0, a.M, kbeg);
  if (VECB) init_ptr<T, BKC, BN>(pb, B, a.ldb, n0, a.N, kbeg);
  // Tiles are loaded in order kt = 0, 1, ...; only the last can be partial.
  auto load = [&](int64_t kt) {
    const int64_t k0 = kbeg + kt * kBK;
    if (kt < nfull) {
      if (VECA) load_full<T, AKC, BM>(ra, pa, AKC ? (int64_t)kBK : kBK * a.lda);
      if (VECB) load_full<T, BKC, BN>(rb, pb, BKC ? (int64_t)kBK : kBK * a.ldb);
    } else {
      if (VECA) load_tail<T, AKC, BM>(ra, pa, a.lda, k0, kend);
      if (VECB) load_tail<T, BKC, BN>(rb, pb, a.ldb, k0, kend);
    }
    if (!VECA) load_tile<T, AKC, BM>(ra, A, a.lda, m0, a.M, k0, kend);
    if (!VECB) load_tile<T, BKC, BN>(rb, B, a.ldb, n0, a.N, k0, kend);
  };
  auto store = [&](int64_t kt, int stage) {
    T* As = lds + stage * LA::SIZE;
    T* Bs = lds + 2 * LA::SIZE + stage * LB::SIZE;
    if (kt < nfull) {
      store_tile<false, T, AKC, BM>(As, ra, 0);
      store_tile<false, T, BKC, BN>(Bs, rb, 0);
    } else {
      const int left = (int)(kend - kbeg - kt * kBK);
      store_tile<true, T, AKC, BM>(As, ra, left);
      store_tile<true, T, BKC, BN>(Bs, rb, left);
    }
  };
  if (ntiles > 0) {
    load(0);
    store(0, 0);
  }
  __syncthreads();
  const bool take_colsum = a.colsum != nullptr && tm == 0 && (int)threadIdx.x < BN;
  double csum = 0.0;
  for (int64_t kt = 0; kt < ntiles; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < ntiles) load(kt + 1);
    const T* As = lds + cur * LA::SIZE;
    const T* Bs = lds + 2 * LA::SIZE + cur * LB::SIZE;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      typename MFT::vec_t fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = read_frag<T, AKC, BM>(As, wm0 + i * MT, ch * kKC, g, c);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[j] = read_frag<T, BKC, BN>(Bs, wn0 + j * MT, ch * kKC, g, c);
#pragma unroll
      for (int s = 0; s < VEC; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = MFT::mma(fa[i][s], fb[j][s], acc[i][j]);
    }
    if (take_colsum) {
      // this thread's column of the B tile: its kBK values in k order, then into
      // the running float64 sum (k past kend was stored as zero)
      T t = T(0);
#pragma unroll
      for (int k = 0; k < kBK; ++k) t = t + (BKC ? Bs[threadIdx.x * LB::STRIDE + k] : Bs[k * LB::STRIDE + threadIdx.x]);
      csum += (double)t;
    }
    if (kt + 1 < ntiles) store(kt + 1, cur ^ 1);
    __syncthreads();
  }
  if (take_colsum) finish_colsum<T>(a, csum, n0 + threadIdx.x, split);
  write_acc<T, TM, TN>(a, acc, m0 + wm0, n0 + wn0, g, c, split, batch);
}

// ---------------------------------------------------------------------------
// Direct global -> LDS loads (global_load_lds_dwordx4: each lane fetches 16
// bytes that land at LDS base + 16 * lane, with no register staging, no LDS
// store instructions and no wait before a store), float32 and float64 alike:
// a k-tile is 64 bytes of k per row (16 floats or 8 doubles), VEC = 16 bytes
// of elements (4 floats or 2 doubles) per vector. Three LDS stages: tile t's
// loads are issued two iterations before it is computed.
// LDS layouts (a 1 KB load instruction fills 1 KB contiguously, so conflicts
// are avoided by choosing which global vector each lane fetches):
//   KC  (k-contiguous operand, BMN rows x 64 bytes): 1 KB chunks of 16 rows;
//       the 16-byte k-vector v of chunk row r sits in 16-byte slot
//       4 r + (v ^ kc_swz(r)), so the 16-byte fragment reads of 16
//       consecutive rows hit distinct banks;
//   MNC (mn-contiguous operand, k-rows of BMN elements): k-row k holds its
//       mn-vectors u at slots u ^ mnc_swz(k), which flips 128 bytes between
//       the k-rows that the two lane groups of a half-wave fragment read
//       (k and k + 4 for float32, k and k + 2 for float64), so they hit
//       different bank halves.
// The 64 x 64 tile has a quarter of the MFMAs to cover a load with, so it keeps
// more tiles in flight.
template <int BM, int BN>
constexpr int kDmaStages = BM == 64 && BN == 64 ? 6 : 3;

__device__ __forceinline__ int kc_swz(int r) { return ((r >> 1) + (r >> 3)) & 3; }
template <typename T>
__device__ __forceinline__ int mnc_swz(int k) {
  return ((k >> (MF<T>::VEC == 4 ? 2 : 1)) & 1) << 3;
}

// Element offset, within one BMN x 64-byte operand tile, of the 16-byte
// vector of (row/col mn, k-vector v) for KC, or of (k-row k, mn-vector u)
// for MNC.
template <typename T>
__device__ __forceinline__ int kc_off(int mn, int v) {
  const int r = mn & 15;
  return (mn >> 4) * (1024 / (int)sizeof(T)) + (4 * r + (v ^ kc_swz(r))) * MF<T>::VEC;
}
template <typename T, int BMN>
__device__ __forceinline__ int mnc_off(int k, int u) {
  return k * BMN + (u ^ mnc_swz<T>(k)) * MF<T>::VEC;
}

// The BMN / 64 load instructions (1 KB each) of each wave per operand tile:
// a wave-uniform base address (the current k-tile's origin, advanced by
// scalar adds) and fixed per-lane 32-bit byte offsets, so issuing a tile
// takes no vector instructions. Offsets are >= 0: clamped rows / columns
// stay at or after the tile origin (the origin is inside the matrix, and
// MN - VEC >= mn0 because MN and mn0 are multiples of VEC).
// An operand that is not 16-byte granular (VECLD false: an odd leading
// dimension, as of a vocabulary of 50257) is fetched 4 bytes per lane instead
// (global_load_lds_dword, 256 bytes of LDS per instruction) into the same
// layout: four times the load instructions, still no vector instruction in the
// loop and no alignment beyond the element's. Each element is then clamped to
// the last row or column by itself, so no vector straddles the edge.
template <typename T, bool KCONTIG, int BMN, bool VECLD>
struct DmaSrc {
  static constexpr int NQ = (VECLD ? 1 : 4) * (BMN / 64);  // instructions per wave
  static constexpr int BYTES = VECLD ? 1024 : 256;         // of LDS per instruction
  const T* base;
  unsigned off[NQ];
  int64_t step;  // elements per k-tile
};

template <typename T, bool KCONTIG, int BMN, bool VECLD>
__device__ __forceinline__ void dma_init(DmaSrc<T, KCONTIG, BMN, VECLD>& s, const T* __restrict__ P, int64_t ld,
                                         int64_t mn0, int64_t MN, int64_t kbeg, int wave, int lane) {
  constexpr int NQ = DmaSrc<T, KCONTIG, BMN, VECLD>::NQ;
  constexpr int VEC = MF<T>::VEC;
  constexpr int RV = BMN / VEC;  // mn-vectors per k-row (MNC)
  s.base = KCONTIG ? P + mn0 * ld + kbeg : P + kbeg * ld + mn0;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int j = wave * NQ + q;  // 1 KB (256-byte) chunk of the tile
    if constexpr (!VECLD) {
      // dword 64 j + lane of the tile: 16-byte slot sl, dword e of it
      const int sl = (64 * j + lane) >> 2, e = lane & 3;
      constexpr int ED = (int)sizeof(T) / 4;  // dwords per element
      if (KCONTIG) {
        const int r = (sl >> 2) & 15;
        int64_t mn = mn0 + (sl >> 2);
        mn = mn < MN ? mn : MN - 1;
        const int v = (sl & 3) ^ kc_swz(r);
        s.off[q] = (unsigned)((mn - mn0) * ld * (int64_t)sizeof(T) + 16 * v + 4 * e);
      } else {
        const int k = sl / RV;
        const int u = (sl % RV) ^ mnc_swz<T>(k);
        int64_t mn = mn0 + VEC * u + e / ED;
        mn = mn < MN ? mn : MN - 1;
        s.off[q] = (unsigned)((k * ld + (mn - mn0)) * (int64_t)sizeof(T) + 4 * (e % ED));
      }
      continue;
    }
    if (KCONTIG) {
      const int r = lane >> 2;
      int64_t mn = mn0 + 16 * j + r;
      mn = mn < MN ? mn : MN - 1;
      const int v = (lane & 3) ^ kc_swz(r);
      s.off[q] = (unsigned)(((mn - mn0) * ld + VEC * v) * (int64_t)sizeof(T));
    } else {
      const int k = (64 * j + lane) / RV;
      const int u = ((64 * j + lane) % RV) ^ mnc_swz<T>(k);
      int64_t mn = mn0 + VEC * u;
      mn = mn < MN ? mn : MN - VEC;
      s.off[q] = (unsigned)((k * ld + (mn - mn0)) * (int64_t)sizeof(T));
    }
  }
  s.step = KCONTIG ? 64 / (int)sizeof(T) : (64 / (int)sizeof(T)) * ld;
}

// Issue one operand tile: chunk q of this wave lands at LDS byte address
// lds_wave + LDS_OFF + 1024 q (lds_wave: wave-uniform, this wave's first
// chunk of stage 0). m0 takes the LDS address one wait state before the load.
// The asm writes no SCC (an s_add here would clobber the carry of a 64-bit
// scalar add the compiler may have split around it): the address is summed
// outside and moved in with s_mov_b32.
template <int LDS_OFF, typename T, bool KCONTIG, int BMN, bool VECLD>
__device__ __forceinline__ void dma_issue(DmaSrc<T, KCONTIG, BMN, VECLD>& s, unsigned lds_wave) {
  typedef DmaSrc<T, KCONTIG, BMN, VECLD> S;
#pragma unroll
  for (int q = 0; q < S::NQ; ++q) {
    const unsigned dst = lds_wave + (unsigned)(LDS_OFF + S::BYTES * q);
    if constexpr (VECLD)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(s.off[q]), "s"(s.base),
                   "s"(dst)
                   : "memory", "m0");
    else
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(s.off[q]), "s"(s.base),
                   "s"(dst)
                   : "memory", "m0");
  }
  s.base += s.step;
}

// This wave's loads except the newest N have landed, then every wave's have.
template <int N>
__device__ __forceinline__ void dma_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int V>
struct IC {
  static constexpr int value = V;
};

// The partial last k-tile through registers, stored in the same layouts
// (k at or past kend as zeros).
template <typename T, bool KCONTIG, int BMN>
__device__ __forceinline__ void dma_tail_store(T* __restrict__ tile, const TileRegs<T, KCONTIG, BMN>& r, int64_t k0,
                                               int64_t kend) {
  using L = TileLayout<T, KCONTIG, BMN>;
  constexpr int VEC = L::VEC;
  constexpr int RV = BMN / VEC;
#pragma unroll
  for (int i = 0; i < L::NVEC; ++i) {
    const int f = threadIdx.x + 256 * i;
    int off;
    int64_t k;
    if (KCONTIG) {
      off = kc_off<T>(f / 4, f % 4);
      k = k0 + (f % 4) * VEC;
    } else {
      off = mnc_off<T, BMN>(f / RV, f % RV);
      k = k0 + f / RV;
    }
    *reinterpret_cast<typename MF<T>::vec_t*>(tile + off) = k < kend ? r.v[i] : typename MF<T>::vec_t(0);
  }
}

// Block tile BM x BN (64 x 64, 128 x 128, or 256 x 128 in float32), 4 waves in a
// 2 x 2 grid of (BM/2) x (BN/2) wave tiles.
template <typename T, int BM, int BN, bool AKC, bool BKC, bool VECA, bool VECB>
__global__ void __launch_bounds__(256, (BM + BN > 384 ? 1 : 2)) gemm_dma_kernel(GemmArgs a) {
  using MFT = MF<T>;
  constexpr int BK = 64 / (int)sizeof(T);
  constexpr int MT = MFT::MT, VEC = MFT::VEC, LV = VEC == 4 ? 2 : 1;  // VEC = 1 << LV
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int TM = WM / MT, TN = WN / MT, NCH = BK / kKC;
  constexpr int TILE_A = BM * BK, TILE_B = BN * BK;  // elements per operand tile
  constexpr int NST = kDmaStages<BM, BN>;
  __shared__ __attribute__((aligned(1024))) T lds[NST * (TILE_A + TILE_B)];

  int tm, tn;
  tile_coords(a, tm, tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int split = blockIdx.y;
  const int64_t batch = blockIdx.z;
  const int64_t kbeg = (int64_t)split * a.k_per_split;
  const int64_t kend = kbeg + a.k_per_split < a.K ? kbeg + a.k_per_split : a.K;
  const T* A = (const T*)a.A + batch * a.sA;
  const T* B = (const T*)a.B + batch * a.sB;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane / MT, c = lane % MT;
  const int wm0 = (wave >> 1) * WM, wn0 = (wave & 1) * WN;

  typename MFT::acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = typename MFT::acc_t(0);

  const int ntiles = kend > kbeg ? (int)((kend - kbeg + BK - 1) / BK) : 0;
  const int nfull = kend > kbeg ? (int)((kend - kbeg) / BK) : 0;
  DmaSrc<T, AKC, BM, VECA> sa;
  DmaSrc<T, BKC, BN, VECB> sb;
  dma_init(sa, A, a.lda, m0, a.M, kbeg, wave, lane);
  dma_init(sb, B, a.ldb, n0, a.N, kbeg, wave, lane);
  auto tileA = [&](int st) { return lds + st * (TILE_A + TILE_B); };
  auto tileB = [&](int st) { return lds + st * (TILE_A + TILE_B) + TILE_A; };
  // LDS byte address of this wave's first A chunk and first B chunk in stage
  // 0 (the low 32 bits of a generic LDS address are the LDS offset)
  const unsigned lds0 = (unsigned)(uintptr_t)lds;
  const unsigned ldsA = __builtin_amdgcn_readfirstlane(lds0 + wave * (BM / 64) * 1024u);
  const unsigned ldsB =
      __builtin_amdgcn_readfirstlane(lds0 + TILE_A * (unsigned)sizeof(T) + wave * (BN / 64) * 1024u);
  constexpr int STAGE_BYTES = (TILE_A + TILE_B) * (int)sizeof(T);
  constexpr int NQT = DmaSrc<T, AKC, BM, VECA>::NQ + DmaSrc<T, BKC, BN, VECB>::NQ;  // loads per wave per k-tile

  // Per-lane fragment offsets within a tile: KC fragment (rows base + c,
  // k-vector (8 / VEC) ch + g); MNC fragment element s (k-row
  // 8 ch + VEC g + s, column base + c).
  auto frag = [&](const T* __restrict__ t, bool kcontig, int bmn, int base, int ch) {
    typename MFT::vec_t v;
    if (kcontig) {
      v = *reinterpret_cast<const typename MFT::vec_t*>(t + kc_off<T>(base + c, (kKC / VEC) * ch + g));
    } else {
      const int n = base + c;
#pragma unroll
      for (int s = 0; s < VEC; ++s) {
        const int k = kKC * ch + VEC * g + s;
        v[s] = t[(bmn == 256   ? mnc_off<T, 256>(k, n >> LV)
               : bmn == 128 ? mnc_off<T, 128>(k, n >> LV)
                            : mnc_off<T, 64>(k, n >> LV)) +
              (n & (VEC - 1))];
      }
    }
    return v;
  };
  const bool take_colsum = a.colsum != nullptr && tm == 0 && (int)threadIdx.x < BN;
  double csum = 0.0;
  auto compute = [&](int st) {
    const T* As = tileA(st);
    const T* Bs = tileB(st);  // st is a constant in the main loop: immediate LDS offsets
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      typename MFT::vec_t fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = frag(As, AKC, BM, wm0 + i * MT, ch);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[j] = frag(Bs, BKC, BN, wn0 + j * MT, ch);
#pragma unroll
      for (int s = 0; s < VEC; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = MFT::mma(fa[i][s], fb[j][s], acc[i][j]);
    }
    if (take_colsum) {
      // this thread's column of the B tile, its BK values in k order, then
      // into the running float64 sum (k past kend was stored as zero)
      const int n = threadIdx.x;
      T t = T(0);
#pragma unroll
      for (int k = 0; k < BK; ++k)
        t = t + (BKC ? Bs[kc_off<T>(n, k >> LV) + (k & (VEC - 1))] : Bs[mnc_off<T, BN>(k, n >> LV) + (n & (VEC - 1))]);
      csum += (double)t;
    }
  };

  auto issue = [&](auto stc) {
    constexpr int st = decltype(stc)::value;
    dma_issue<st * STAGE_BYTES>(sa, ldsA);
    dma_issue<st * STAGE_BYTES>(sb, ldsB);
  };
  // One k-tile: this wave's loads of tile kt have landed (the NST - 2 tiles
  // after it may still be in flight), then every wave's have, and every wave is
  // done with the stage about to be refilled (that of tile kt - 1); then the
  // loads of tile kt + NST - 1 and the MFMAs of tile kt. The conditions have the
  // form of the main loop's, so that those it implies fold away there (as
  // nfull - 1 - kt >= ... each cost a branch a step: 8192 x 512 x 2048 130 -> 143 us).
  auto step = [&](auto stc, int kt) {
    constexpr int st = decltype(stc)::value;
    if (kt + NST - 2 < nfull)
      dma_wait_barrier<(NST - 2) * NQT>();
    else if (NST > 5 && kt + 3 < nfull)
      dma_wait_barrier<(NST > 5 ? 3 : 0) * NQT>();
    else if (NST > 4 && kt + 2 < nfull)
      dma_wait_barrier<(NST > 4 ? 2 : 0) * NQT>();
    else if (NST > 3 && kt + 1 < nfull)
      dma_wait_barrier<(NST > 3 ? 1 : 0) * NQT>();
    else
      dma_wait_barrier<0>();
    if (kt + NST - 1 < nfull) issue(IC<(st + NST - 1) % NST>());
    compute(st);
  };
  auto each_stage = [&](auto f) {  // f(IC<0>), ..., f(IC<NST - 1>)
    [&]<int... I>(std::integer_sequence<int, I...>) { (f(IC<I>()), ...); }(std::make_integer_sequence<int, NST>());
  };
  static_assert(NST >= 3 && NST <= 6 && (NST - 2) * NQT < 64, "waits of step(), vmcnt range");
  // The three-stage kernels' steps are written out: run through each_stage they
  // are the same instructions, but 8192 x 512 x 2048 took 146 us (137 written out)
  // at the same cycle count, that is at a lower clock.
  if constexpr (NST == 3) {
    if (nfull > 0) issue(IC<0>());
    if (nfull > 1) issue(IC<1>());
  } else {
    each_stage([&](auto stc) {
      constexpr int st = decltype(stc)::value;
      if (st < NST - 1 && st < nfull) issue(stc);
    });
  }
  // A long range without a K split is summed in pieces (a.fold_groups): a chain
  // of thousands of float32 additions would lose what the splits of the 128-wide
  // tiles keep. 32 vector instructions per 192 k beside 96 MFMAs, no difference
  // in time that could be measured (1186 and 1188 us a block at 5 x 499 x 768).
  constexpr bool FOLD = BM == 64;
  typename MFT::acc_t tot[FOLD ? TM : 1][FOLD ? TN : 1];
  if constexpr (FOLD)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) tot[i][j] = typename MFT::acc_t(0);
  auto fold = [&]() {
    if constexpr (FOLD)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          tot[i][j] += acc[i][j];
          acc[i][j] = typename MFT::acc_t(0);
        }
  };
  int kt = 0, grp = 0;
  for (; kt + NST <= nfull; kt += NST) {
    if constexpr (NST == 3) {
      step(IC<0>(), kt);
      step(IC<1>(), kt + 1);
      step(IC<2>(), kt + 2);
    } else {
      each_stage([&](auto stc) { step(stc, kt + decltype(stc)::value); });
    }
    if constexpr (FOLD)
      if (++grp == a.fold_groups) {
        fold();
        grp = 0;
      }
  }
  if constexpr (NST == 3) {
    if (kt < nfull) step(IC<0>(), kt);
    if (kt + 1 < nfull) step(IC<1>(), kt + 1);
  } else {
    each_stage([&](auto stc) {
      if (kt + decltype(stc)::value < nfull) step(stc, kt + decltype(stc)::value);
    });
  }
  const int st = nfull % NST;  // stage of the partial tile, if any
  if (ntiles > nfull) {  // the partial last k-tile, through registers
    const int64_t k0 = kbeg + (int64_t)nfull * BK;
    TileRegs<T, AKC, BM> ra;
    TileRegs<T, BKC, BN> rb;
    if constexpr (VECA) {
      TilePtr<T, AKC, BM> pa;
      init_ptr<T, AKC, BM>(pa, A, a.lda, m0, a.M, k0);
      load_tail<T, AKC, BM>(ra, pa, a.lda, k0, kend);
    } else {
      load_tile<T, AKC, BM>(ra, A, a.lda, m0, a.M, k0, kend);
    }
    if constexpr (VECB) {
      TilePtr<T, BKC, BN> pb;
      init_ptr<T, BKC, BN>(pb, B, a.ldb, n0, a.N, k0);
      load_tail<T, BKC, BN>(rb, pb, a.ldb, k0, kend);
    } else {
      load_tile<T, BKC, BN>(rb, B, a.ldb, n0, a.N, k0, kend);
    }
    __syncthreads();  // every wave is done with the stage being refilled
    dma_tail_store<T, AKC, BM>(tileA(st), ra, k0, kend);
    dma_tail_store<T, BKC, BN>(tileB(st), rb, k0, kend);
    __syncthreads();
    compute(st);
  }
  if constexpr (FOLD)
    if (a.fold_groups > 0)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += tot[i][j];
  if (take_colsum) finish_colsum<T>(a, csum, n0 + threadIdx.x, split);
  write_acc<T, TM, TN, true>(a, acc, m0 + wm0, n0 + wn0, g, c, split, batch);
}

template <typename T, int BM, int BN, bool AKC, bool BKC>
static void launch_variant(const GemmArgs& a, dim3 grid, bool veca, bool vecb, bool dma) {
  if (!dma) {
    if constexpr (BM == 128 && BN == 128) {  // the other tiles: gemm_dma_kernel only (see gemm_impl)
      if (veca && vecb)
        gemm_kernel<T, BM, BN, AKC, BKC, true, true><<<grid, 256, 0, stream()>>>(a);
      else if (veca)
        gemm_kernel<T, BM, BN, AKC, BKC, true, false><<<grid, 256, 0, stream()>>>(a);
      else if (vecb)
        gemm_kernel<T, BM, BN, AKC, BKC, false, true><<<grid, 256, 0, stream()>>>(a);
      else
        gemm_kernel<T, BM, BN, AKC, BKC, false, false><<<grid, 256, 0, stream()>>>(a);
    }
  } else if (veca && vecb) {
    gemm_dma_kernel<T, BM, BN, AKC, BKC, true, true><<<grid, 256, 0, stream()>>>(a);
  } else if (veca) {
    gemm_dma_kernel<T, BM, BN, AKC, BKC, true, false><<<grid, 256, 0, stream()>>>(a);
  } else if (vecb) {
    gemm_dma_kernel<T, BM, BN, AKC, BKC, false, true><<<grid, 256, 0, stream()>>>(a);
  } else {
    gemm_dma_kernel<T, BM, BN, AKC, BKC, false, false><<<grid, 256, 0, stream()>>>(a);
  }
}

template <typename T, int BM, int BN>
void launch_layout(const GemmArgs& a, dim3 grid, int akc, int bkc, bool veca, bool vecb, bool dma) {
  if (akc && bkc)
    launch_variant<T, BM, BN, true, true>(a, grid, veca, vecb, dma);
  else if (akc)
    launch_variant<T, BM, BN, true, false>(a, grid, veca, vecb, dma);
  else if (bkc)
    launch_variant<T, BM, BN, false, true>(a, grid, veca, vecb, dma);
  else
    launch_variant<T, BM, BN, false, false>(a, grid, veca, vecb, dma);
}

}  // namespace dtmi
