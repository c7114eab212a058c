// Device kernels of the solve phase: CSR SpMV / SpMM with fused smoother
// epilogues, reductions with a last-block finish, and the dense coarse solve.
//
// Layout: vectors with k right-hand sides are row-major (n x k), so the k
// values of one vertex are contiguous and a gather x[col*k + c] by k lanes is
// one coalesced access.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fem_internal.hpp"

namespace fem {

constexpr int kNT = 256;  // threads per block of the solve kernels

enum SpmvMode : int {
  kAssign = 0,   // y = A x
  kResid = 1,    // y = b - A x
  kAdd = 2,      // y += A x
  kJacobi = 3,   // xn = x + c1 * dinv * (b - A x)
  kCheb = 4,     // r = dinv (b - A x); d = c1 d + c2 r; xn = x + d
  kAssignScale = 5,  // y = A x; xn = c1 * dinv * y; d = xn when d != null (a
                     // restriction that also takes the next level's first
                     // smoothing step from zero)
};

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own
// L2.  Gathering kernels remap the hardware block index so that XCD j runs a
// contiguous range of logical blocks: neighbouring rows (Morton order) then
// share one L2 and the gathered vector is fetched from HBM about once
// instead of once per XCD.  A bijection of [0, nblocks) for any nblocks.
constexpr unsigned kNumXcd = 8;

__device__ __forceinline__ unsigned xcd_block(unsigned bid, unsigned nblocks) {
  const unsigned x = bid % kNumXcd, i = bid / kNumXcd;
  const unsigned q = nblocks / kNumXcd, r = nblocks % kNumXcd;
  return x * q + min(x, r) + i;
}

// Rows of a block in a loop over n rows, `per` rows per block and pass, laid
// out so that each XCD sweeps one contiguous range of rows with a single
// front: the blocks of one XCD take consecutive groups of `per` rows of its
// range, then all advance together by (its blocks) x per.  Contiguous chunks
// per block instead give each XCD hundreds of separate fronts whose gathered
// neighbourhoods do not fit its L2 (measured for 16 FP64 columns at 161^3:
// 3.2x the algorithmic HBM reads).  The XCD ranges are those of the
// contiguous logical blocks xcd_block assigns to it, so the rows are covered
// once for any grid size.
struct XcdRows {
  int64_t hi;     // end of this XCD's rows
  int64_t first;  // first row group of this block
  int64_t step;   // rows between its groups
};

__device__ __forceinline__ XcdRows xcd_rows(int64_t n, int64_t per) {
  const unsigned nb = gridDim.x, bid = blockIdx.x;
  const unsigned x = bid % kNumXcd, i = bid / kNumXcd;
  const unsigned q = nb / kNumXcd, r = nb % kNumXcd;
  const unsigned nbx = q + (x < r ? 1u : 0u);  // blocks on this XCD
  const unsigned lb0 = x * q + min(x, r);      // their first logical block
  const int64_t chunk = ((n + nb - 1) / nb + per - 1) / per * per;
  const int64_t lo = (int64_t)lb0 * chunk;
  XcdRows R;
  R.hi = min(n, (int64_t)(lb0 + nbx) * chunk);
  R.first = lo + (int64_t)i * per;
  R.step = (int64_t)nbx * per;
  return R;
}

// Matrix entries are read once per SpMV: nontemporal loads keep them from
// evicting the gathered vector from L2 (measured: -15 % time at 4.2M rows).
template <typename T>
__device__ __forceinline__ T ntload(const T* p) {
  return __builtin_nontemporal_load(p);
}

template <typename T>
__device__ __forceinline__ T shfl_xor_t(T v, int mask, int width) {
  return __shfl_xor(v, mask, width);
}

// One epilogue for all modes; `acc` = (A x)_row for column c.
template <int MODE, typename T, typename V>
__device__ __forceinline__ void spmv_epilogue(int64_t idx, int64_t row, T acc, T* __restrict__ y,
                                              const T* __restrict__ x, const T* __restrict__ b,
                                              const V* __restrict__ dinv, T* __restrict__ d,
                                              T* __restrict__ xn, T c1, T c2) {
  if (MODE == kAssign) {
    y[idx] = acc;
  } else if (MODE == kAssignScale) {
    y[idx] = acc;
    const T v = c1 * (T)dinv[row] * acc;
    xn[idx] = v;
    if (d) d[idx] = v;
  } else if (MODE == kResid) {
    y[idx] = b[idx] - acc;
  } else if (MODE == kAdd) {
    y[idx] += acc;
  } else if (MODE == kJacobi) {
    xn[idx] = x[idx] + c1 * (T)dinv[row] * (b[idx] - acc);
  } else {  // kCheb: b, D^-1 and d are read once; nontemporal for FP64 (measured faster there, not for FP32)
    constexpr bool nt = sizeof(T) == 8;
    T r = (T)(nt ? ntload(dinv + row) : dinv[row]) * ((nt ? ntload(b + idx) : b[idx]) - acc);
    T dn = (c1 != T(0) ? c1 * (nt ? ntload(d + idx) : d[idx]) : T(0)) + c2 * r;
    d[idx] = dn;
    xn[idx] = x[idx] + dn;
  }
}

// The same for one column and V = T in two halves, so that the row's vector
// entries can be loaded ahead of the row sum (same values, same order).
template <typename T>
struct SpmvRow {
  T sd, x, b, dinv, d, y;

  template <int MODE>
  __device__ __forceinline__ void load(int64_t row, const T* __restrict__ sdp, const T* __restrict__ xp,
                                       const T* __restrict__ yp, const T* __restrict__ bp,
                                       const T* __restrict__ dinvp, const T* __restrict__ dp, T c1) {
    constexpr bool nt = MODE == kCheb && sizeof(T) == 8;
    if (sdp) sd = sdp[row];
    if (sdp || MODE == kJacobi || MODE == kCheb) x = xp[row];
    if (MODE == kResid || MODE == kJacobi || MODE == kCheb) b = nt ? ntload(bp + row) : bp[row];
    if (MODE == kAssignScale || MODE == kJacobi || MODE == kCheb) dinv = nt ? ntload(dinvp + row) : dinvp[row];
    if (MODE == kCheb) d = c1 != T(0) ? (nt ? ntload(dp + row) : dp[row]) : T(0);
    if (MODE == kAdd) y = yp[row];
  }

  // returns the row's result; LAST: a smoother's last step, d is not needed
  template <int MODE, bool LAST = false>
  __device__ __forceinline__ T store(int64_t row, T acc, T* __restrict__ yp, T* __restrict__ dp,
                                     T* __restrict__ xn, T c1, T c2) {
    T out = acc;
    if (MODE == kAssign) {
      yp[row] = out;
    } else if (MODE == kAssignScale) {
      yp[row] = acc;
      out = c1 * dinv * acc;
      xn[row] = out;
      if (dp) dp[row] = out;
    } else if (MODE == kResid) {
      yp[row] = out = b - acc;
    } else if (MODE == kAdd) {
      yp[row] = out = y + acc;
    } else if (MODE == kJacobi) {
      xn[row] = out = x + c1 * dinv * (b - acc);
    } else {
      const T r = dinv * (b - acc);
      const T dn = (c1 != T(0) ? c1 * d : T(0)) + c2 * r;
      if (!LAST) dp[row] = dn;
      xn[row] = out = x + dn;
    }
    return out;
  }
};

// Single right-hand side: G lanes per row, strided over the row's entries,
// reduced by a butterfly (fixed order).  A lane's entries go in batches of four
// (two dependent waits on memory for four entries instead of for each): 49^3
// FP64 level 1 (5,500 rows, Chebyshev) 4.4 -> 3.4 us, its restriction (200 rows)
// 8.3 -> 4.7; 161^3 FP32 level 2 5.6 -> 4.9.
constexpr int kCsrBatch = 4;
template <typename V, typename T, int G, int MODE>
__global__ void __launch_bounds__(kNT) csr_vec_kernel(int64_t n, const int32_t* __restrict__ rp,
                                                    const int32_t* __restrict__ ci, const V* __restrict__ val,
                                                    const T* __restrict__ x, T* __restrict__ y,
                                                    const T* __restrict__ b, const V* __restrict__ dinv,
                                                    T* __restrict__ d, T* __restrict__ xn, T c1, T c2) {
  const int64_t row = ((int64_t)xcd_block(blockIdx.x, gridDim.x) * kNT + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  if (row >= n) return;
  const int s = rp[row], e = rp[row + 1];
  T acc = T(0);
  for (int k = s + lane; k < e; k += kCsrBatch * G) {
    int c[kCsrBatch];
    T v[kCsrBatch], xv[kCsrBatch];
#pragma unroll
    for (int j = 0; j < kCsrBatch; ++j) {
      if (k + j * G < e) {
        c[j] = ntload(ci + k + j * G);
        v[j] = (T)ntload(val + k + j * G);
      }
    }
#pragma unroll
    for (int j = 0; j < kCsrBatch; ++j)
      if (k + j * G < e) xv[j] = x[c[j]];
#pragma unroll
    for (int j = 0; j < kCsrBatch; ++j)
      if (k + j * G < e) acc += v[j] * xv[j];
  }
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) acc += shfl_xor_t(acc, off, G);
  if (lane == 0) spmv_epilogue<MODE, T, V>(row, row, acc, y, x, b, dinv, d, xn, c1, c2);
}

// Sliced ELL, one RHS: a wavefront owns a slice of 64 rows, lane = row; the
// slice is column-major so every step k is one coalesced 64-wide load of
// values and of columns, and the k steps are independent loads the compiler
// keeps in flight together.  Sequential per-row sum (fixed order).
struct SellView {
  const int32_t* sp;    // nslices + 1 element offsets
  const int32_t* sc;    // int32 columns
  const uint16_t* sc16; // 16-bit column codes of compact slices
  const int32_t* swin;  // kSellWindows window bases per slice (-1: not compact)
  const int32_t* srow;  // row at each position (null: position = row)
  const double* sd64;   // diagonal outside the slices (null: in the slices)
  const float* sd32;
};

inline SellView sell_view(const Csr& A) {
  return SellView{A.sp.get(), A.sc.get(), A.sc16.get(), A.swin.get(), A.srow.size() ? A.srow.get() : nullptr,
                  A.sd64.size() ? A.sd64.get() : nullptr, A.sd32.size() ? A.sd32.get() : nullptr};
}

// the diagonal held outside the slices, in the working precision (null when
// the slices hold it)
template <typename T>
__device__ __forceinline__ const T* sell_diag(const SellView& S);
template <>
__device__ __forceinline__ const double* sell_diag<double>(const SellView& S) { return S.sd64; }
template <>
__device__ __forceinline__ const float* sell_diag<float>(const SellView& S) { return S.sd32; }

// Window bases of a compact slice, read once per wavefront into scalar
// registers (named members, not an array: the select tree below must stay
// register selects).
struct SellWin {
  int b0, b1, b2, b3, b4, b5, b6, b7;
};

__device__ __forceinline__ int sell_col(unsigned c, SellWin W) {
  const bool s0 = c & (1u << kSellWinBits), s1 = c & (2u << kSellWinBits), s2 = c & (4u << kSellWinBits);
  const int lo = s1 ? (s0 ? W.b3 : W.b2) : (s0 ? W.b1 : W.b0);
  const int hi = s1 ? (s0 ? W.b7 : W.b6) : (s0 ? W.b5 : W.b4);
  return (s2 ? hi : lo) + (int)(c & ((1u << kSellWinBits) - 1u));
}

// value of a stored matrix entry: FP64 / FP32 as stored, FP16 kept as its
// 16-bit pattern (uint16_t)
template <typename T, typename V>
__device__ __forceinline__ T sell_val(const V* p) {
  return (T)ntload(p);
}
template <>
__device__ __forceinline__ float sell_val<float, uint16_t>(const uint16_t* p) {
  return (float)__builtin_bit_cast(_Float16, ntload(p));
}

// Steps k .. k + N - 1 of a lane's entries added to acc in entry order; steps
// from w (wave-uniform) on read entry w - 1 again and add nothing, without
// branches between the loads.
template <int N, typename T, typename V, typename C, typename Col>
__device__ __forceinline__ T sell_batch(T acc, int k, int w, const C* __restrict__ cp, const V* __restrict__ vp,
                                        const T* __restrict__ x, Col& col) {
  C c[N];
  T v[N], xv[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int e = 64 * (k + j < w ? k + j : w - 1);
    c[j] = ntload(cp + e);
    v[j] = sell_val<T>(vp + e);
  }
#pragma unroll
  for (int j = 0; j < N; ++j) xv[j] = x[col(c[j])];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const T s = acc + v[j] * xv[j];
    acc = k + j < w ? s : acc;
  }
  return acc;
}

// Sum of w steps of a lane's entries, in entry order.  A batch is two dependent
// waits on memory (columns and values, then x) whatever its length, so eight
// steps share them, the last seven or fewer too.  Against batches of four and
// single last steps, the row's vector entries loaded after the sum (Chebyshev
// step): 1003 x 701 levels 1 and 2 (53,610 and 4,000 rows) 7.0 and 7.3 -> 5.0
// and 5.4 us, 97^3 level 1 (43,000 rows, 4 lanes each) 8.6 -> 6.6 us.  Level-0
// restrictions in 3D (88 entries a row, 8 lanes) are bound by the lines their
// gathers touch: 42.0 -> 40.5 us at 161^3.
constexpr int kSellBatch = 8;
template <typename T, typename V, typename C, typename Col>
__device__ __forceinline__ T sell_batches(int w, const C* __restrict__ cp, const V* __restrict__ vp,
                                          const T* __restrict__ x, Col&& col) {
  T acc = T(0);
  int k = 0;
  for (; k + kSellBatch <= w; k += kSellBatch) acc = sell_batch<kSellBatch, T, V>(acc, k, w, cp, vp, x, col);
  if (w - k > 4)
    acc = sell_batch<kSellBatch, T, V>(acc, k, w, cp, vp, x, col);
  else if (w - k > 0)
    acc = sell_batch<4, T, V>(acc, k, w, cp, vp, x, col);
  return acc;
}

// Row sum of slice `slice` (wave-uniform) for this lane's row.  Compact
// slices read 2-byte column codes: bits 13-15 select one of the slice's 8
// window bases, bits 0-12 are the offset.
template <typename T, typename V = T>
__device__ __forceinline__ T sell_row_sum(const SellView& S, int slice, int lane, const V* __restrict__ sv,
                                          const T* __restrict__ x) {
  const int off = __builtin_amdgcn_readfirstlane(S.sp[slice]);
  const int w = __builtin_amdgcn_readfirstlane((S.sp[slice + 1] - off) >> 6);
  const V* vp = sv + off + lane;
  static_assert(kSellWindows == 8, "sell_col selects among 8 windows");
  const int32_t* wp = S.swin + slice * kSellWindows;
  const SellWin W{__builtin_amdgcn_readfirstlane(wp[0]), __builtin_amdgcn_readfirstlane(wp[1]),
                  __builtin_amdgcn_readfirstlane(wp[2]), __builtin_amdgcn_readfirstlane(wp[3]),
                  __builtin_amdgcn_readfirstlane(wp[4]), __builtin_amdgcn_readfirstlane(wp[5]),
                  __builtin_amdgcn_readfirstlane(wp[6]), __builtin_amdgcn_readfirstlane(wp[7])};
  if (W.b0 >= 0)
    return sell_batches<T, V>(w, S.sc16 + off + lane, vp, x, [&](unsigned c) { return sell_col(c, W); });
  return sell_batches<T, V>(w, S.sc + off + lane, vp, x, [](int c) { return c; });
}

// ---- LDS-staged sliced ELL (one lane per row, row order) ------------------------
// A block of L.bs consecutive slices first copies x at the distinct columns
// its rows use into LDS (one global gather per distinct column instead of
// one per stored entry: 0.18 per entry at 161^3 with 8 slices), then reads
// the entries' x from LDS through 16-bit indices.
struct LdsView {
  int bs;                // slices per block
  const uint16_t* lc;    // LDS index per stored entry
  const int32_t* lcs;    // block offsets into lcols
  const int32_t* lcols;  // distinct columns per block, ascending
};

inline LdsView lds_view(const LdsList& l) { return LdsView{l.bs, l.lc.get(), l.lcs.get(), l.lcols.get()}; }

// x at the block's distinct columns into xs (then a block barrier), in two
// halves: the first kStageCols columns of each thread are loaded by begin(),
// so that loads which do not depend on them can be issued before finish()
// gathers x.
constexpr int kStageCols = 4;
struct LdsStage {
  int c0, nc;
  int col[kStageCols];

  __device__ __forceinline__ void begin(const LdsView& L, unsigned blk) {
    c0 = L.lcs[blk];
    nc = L.lcs[blk + 1] - c0;
#pragma unroll
    for (int j = 0; j < kStageCols; ++j) {
      const int t = (int)threadIdx.x + j * (int)blockDim.x;
      if (t < nc) col[j] = L.lcols[c0 + t];
    }
  }

  template <typename T>
  __device__ __forceinline__ void finish(const LdsView& L, const T* __restrict__ x, T* xs) {
    T v[kStageCols];
#pragma unroll
    for (int j = 0; j < kStageCols; ++j)
      if ((int)threadIdx.x + j * (int)blockDim.x < nc) v[j] = x[col[j]];
#pragma unroll
    for (int j = 0; j < kStageCols; ++j) {
      const int t = (int)threadIdx.x + j * (int)blockDim.x;
      if (t < nc) xs[t] = v[j];
    }
    for (int t = (int)threadIdx.x + kStageCols * (int)blockDim.x; t < nc; t += blockDim.x)
      xs[t] = x[L.lcols[c0 + t]];
    __syncthreads();
  }
};

// The first HEAD steps of a lane's row (LDS indices and stored values),
// loaded before the staging barrier: they do not depend on x, so their memory
// latency runs beside the staging's (list offsets -> columns -> x) instead of
// after it.  In groups of four, and the remainder of a row that ends there;
// which loads are issued is the same for the whole wavefront.  The steps after
// the head go in batches of eight.  HEAD kLdsBatch: no head, batches of eight;
// 0: no head, batches of four (fewest registers).
constexpr int kLdsBatch = -8;
template <typename V, int HEAD>
struct SliceHead {
  unsigned c[HEAD > 0 ? HEAD : 1], rc[3];
  V v[HEAD > 0 ? HEAD : 1], rv[3];
  int off, w;  // the slice's first element and steps
};

template <typename V, int HEAD>
__device__ __forceinline__ void lds_head(SliceHead<V, HEAD>& H, const SellView& S, const LdsView& L, int slice,
                                         int lane, const V* __restrict__ sv) {
  H.off = __builtin_amdgcn_readfirstlane(S.sp[slice]);
  H.w = __builtin_amdgcn_readfirstlane((S.sp[slice + 1] - H.off) >> 6);
  const V* vp = sv + H.off + lane;
  const uint16_t* cp = L.lc + H.off + lane;
#pragma unroll
  for (int g = 0; g < HEAD; g += 4) {
    if (g + 4 <= H.w) {
#pragma unroll
      for (int j = g; j < g + 4; ++j) {
        H.c[j] = ntload(cp + 64 * j);
        H.v[j] = ntload(vp + 64 * j);
      }
    }
  }
  if (H.w < HEAD) {
    const int base = H.w & ~3;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      if (base + j < H.w) {
        H.rc[j] = ntload(cp + 64 * (base + j));
        H.rv[j] = ntload(vp + 64 * (base + j));
      }
    }
  }
}

// value of a stored matrix entry in the working precision: FP64 / FP32 as
// stored, FP16 kept as its 16-bit pattern (uint16_t)
template <typename T, typename V>
__device__ __forceinline__ T sell_cvt(V v) { return (T)v; }
template <>
__device__ __forceinline__ float sell_cvt<float, uint16_t>(uint16_t v) {
  return (float)__builtin_bit_cast(_Float16, v);
}

// row sum with x from LDS, the head's entries first (same entry order as
// sell_row_sum)
template <typename T, typename V, int HEAD>
__device__ __forceinline__ T lds_row_sum(const SliceHead<V, HEAD>& H, const LdsView& L, int lane,
                                         const V* __restrict__ sv, const T* xs) {
  T acc = T(0);
#pragma unroll
  for (int g = 0; g < HEAD; g += 4) {
    if (g + 4 <= H.w) {
#pragma unroll
      for (int j = g; j < g + 4; ++j) acc += sell_cvt<T>(H.v[j]) * xs[H.c[j]];
    }
  }
  if (H.w < HEAD) {
    const int base = H.w & ~3;
#pragma unroll
    for (int j = 0; j < 3; ++j)
      if (base + j < H.w) acc += sell_cvt<T>(H.rv[j]) * xs[H.rc[j]];
    return acc;
  }
  const V* vp = sv + H.off + lane;
  const uint16_t* cp = L.lc + H.off + lane;
  if constexpr (HEAD != 0) {
    auto col = [](unsigned c) { return c; };
    int k = HEAD > 0 ? HEAD : 0;
    for (; k + kSellBatch <= H.w; k += kSellBatch)
      acc = sell_batch<kSellBatch, T, V>(acc, k, H.w, cp, vp, xs, col);
    if (k < H.w) acc = sell_batch<kSellBatch, T, V>(acc, k, H.w, cp, vp, xs, col);
    return acc;
  }
  int k = 0;
  for (; k + 4 <= H.w; k += 4) {
    unsigned c[4];
    V v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      c[j] = ntload(cp + 64 * (k + j));
      v[j] = ntload(vp + 64 * (k + j));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) acc += sell_cvt<T>(v[j]) * xs[c[j]];
  }
  for (; k < H.w; ++k) acc += sell_cvt<T>(ntload(vp + 64 * k)) * xs[ntload(cp + 64 * k)];
  return acc;
}

// A block on the LDS-staged copy: L.bs slices, a wavefront each (blocks of
// more wavefronts use the others for staging only).
constexpr int kLdsMaxSlices = 8;
constexpr int kLdsMaxNT = 64 * kLdsMaxSlices;

struct LdsWave {
  int lane, slice;
  bool live;    // this wavefront has a slice
  bool on;      // and this lane one of its rows
  int64_t pos;  // the lane's row position
};

__device__ __forceinline__ LdsWave lds_wave(const LdsView& L, unsigned blk, int64_t n, int64_t nslices) {
  LdsWave w;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  w.lane = threadIdx.x & 63;
  w.slice = (int)blk * L.bs + wv;
  w.live = wv < L.bs && w.slice < nslices;
  w.pos = (int64_t)w.slice * 64 + w.lane;
  w.on = w.live && w.pos < n;
  return w;
}

// SpMV with the fused epilogues on the LDS-staged copy; grid = one block per
// L.bs slices, dynamic LDS = the largest distinct-column count x sizeof(T).
// The row's vector entries are loaded before the staging barrier too.
template <typename T, int MODE, int HEAD>
__global__ void __launch_bounds__(kLdsMaxNT) sell_lds_kernel(int64_t n, int64_t nslices, SellView S, LdsView L,
                                                           const T* __restrict__ sv, const T* __restrict__ x,
                                                           T* __restrict__ y, const T* __restrict__ b,
                                                           const T* __restrict__ dinv, T* __restrict__ d,
                                                           T* __restrict__ xn, T c1, T c2) {
  extern __shared__ unsigned char lds_raw[];
  T* xs = reinterpret_cast<T*>(lds_raw);
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const LdsWave w = lds_wave(L, blk, n, nslices);
  const T* sd = sell_diag<T>(S);
  LdsStage G;
  SliceHead<T, HEAD> H;
  SpmvRow<T> R;
  int64_t row = w.pos;
  G.begin(L, blk);
  if (w.live) lds_head(H, S, L, w.slice, w.lane, sv);
  if (w.on) {
    if (S.srow) row = S.srow[w.pos];
    R.template load<MODE>(row, sd, x, y, b, dinv, d, c1);
  }
  G.finish<T>(L, x, xs);
  if (!w.on) return;
  T acc = lds_row_sum<T>(H, L, w.lane, sv, xs);
  if (sd) acc += R.sd * R.x;  // the diagonal term, last
  R.template store<MODE>(row, acc, y, d, xn, c1, c2);
}

// G lanes per row (slices of 64 / G rows): each lane sums its strided share
// of the row, then a butterfly over the G lanes adds the shares (fixed order).
template <typename T, int MODE, int G = 1>
__global__ void __launch_bounds__(kNT) sell_kernel(int64_t n, int64_t nslices, SellView S, const T* __restrict__ sv,
                                                 const T* __restrict__ x, T* __restrict__ y,
                                                 const T* __restrict__ b, const T* __restrict__ dinv,
                                                 T* __restrict__ d, T* __restrict__ xn, T c1, T c2) {
  // the slice index is the same on every lane of the wavefront
  const int slice =
      __builtin_amdgcn_readfirstlane((int)(xcd_block(blockIdx.x, gridDim.x) * (kNT / 64) + (threadIdx.x >> 6)));
  const int lane = threadIdx.x & 63;
  if (slice >= nslices) return;
  // the row's vector entries are loaded beside the first entries
  const int64_t pos = (int64_t)slice * (64 / G) + lane / G;
  const bool on = (G == 1 || (lane & (G - 1)) == 0) && pos < n;
  const T* sd = sell_diag<T>(S);
  int64_t row = pos;
  SpmvRow<T> R;
  if (on) {
    if (S.srow) row = S.srow[pos];
    R.template load<MODE>(row, sd, x, y, b, dinv, d, c1);
  }
  T acc = sell_row_sum<T>(S, slice, lane, sv, x);
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) acc += shfl_xor_t(acc, off, G);
  if (!on) return;
  if (sd) acc += R.sd * R.x;  // the diagonal term, last
  R.template store<MODE>(row, acc, y, d, xn, c1, c2);
}

// k right-hand sides with k a multiple of VW = 16 / sizeof(T): L lanes per
// row, each lane owns VW consecutive columns and gathers them as one 16-byte
// load (measured for k = 16 FP32 at 161^3: 1.6x the one-column-per-lane kernel).
template <typename T, int L, int MODE>
__global__ void __launch_bounds__(kNT) csr_multi_vec_kernel(int64_t n, int k, const int32_t* __restrict__ rp,
                                                          const int32_t* __restrict__ ci, const T* __restrict__ val,
                                                          const T* __restrict__ x, T* __restrict__ y,
                                                          const T* __restrict__ b, const T* __restrict__ dinv,
                                                          T* __restrict__ d, T* __restrict__ xn, T c1, T c2) {
  constexpr int VW = 16 / (int)sizeof(T);
  typedef T vec __attribute__((ext_vector_type(VW)));
  const int64_t row = ((int64_t)xcd_block(blockIdx.x, gridDim.x) * kNT + threadIdx.x) / L;
  const int c0 = (int)(threadIdx.x & (L - 1)) * VW;
  if (row >= n || c0 >= k) return;
  const int s = rp[row], e = rp[row + 1];
  vec acc = (vec)(T(0));
  int q = s;
  for (; q + 4 <= e; q += 4) {
    const int j0 = ci[q], j1 = ci[q + 1], j2 = ci[q + 2], j3 = ci[q + 3];
    const T v0 = val[q], v1 = val[q + 1], v2 = val[q + 2], v3 = val[q + 3];
    const vec g0 = *(const vec*)(x + (int64_t)j0 * k + c0), g1 = *(const vec*)(x + (int64_t)j1 * k + c0);
    const vec g2 = *(const vec*)(x + (int64_t)j2 * k + c0), g3 = *(const vec*)(x + (int64_t)j3 * k + c0);
    acc += v0 * g0;
    acc += v1 * g1;
    acc += v2 * g2;
    acc += v3 * g3;
  }
  for (; q < e; ++q) acc += val[q] * *(const vec*)(x + (int64_t)ci[q] * k + c0);
  const int64_t idx = row * k + c0;
  if (MODE == kAssign) {
    *(vec*)(y + idx) = acc;
  } else if (MODE == kAssignScale) {
    *(vec*)(y + idx) = acc;
    const vec v = (c1 * (T)dinv[row]) * acc;
    *(vec*)(xn + idx) = v;
    if (d) *(vec*)(d + idx) = v;
  } else if (MODE == kResid) {
    *(vec*)(y + idx) = *(const vec*)(b + idx) - acc;
  } else if (MODE == kAdd) {
    *(vec*)(y + idx) += acc;
  } else if (MODE == kJacobi) {
    *(vec*)(xn + idx) = *(const vec*)(x + idx) + (c1 * dinv[row]) * (*(const vec*)(b + idx) - acc);
  } else {  // kCheb
    const vec r = dinv[row] * (*(const vec*)(b + idx) - acc);
    const vec dn = (c1 != T(0) ? c1 * *(const vec*)(d + idx) : (vec)(T(0))) + c2 * r;
    *(vec*)(d + idx) = dn;
    *(vec*)(xn + idx) = *(const vec*)(x + idx) + dn;
  }
}

// k right-hand sides, long rows: as csr_multi_vec_kernel, and ES lane groups
// split the row's entries (group e takes entries e, e + ES, ...); a butterfly
// over the groups adds their sums (fixed order).  L * ES lanes per row.
template <typename T, int L, int ES, int MODE>
__global__ void __launch_bounds__(kNT) csr_multi_split_kernel(int64_t n, int k, const int32_t* __restrict__ rp,
                                                            const int32_t* __restrict__ ci,
                                                            const T* __restrict__ val, const T* __restrict__ x,
                                                            T* __restrict__ y, const T* __restrict__ b,
                                                            const T* __restrict__ dinv, T* __restrict__ d,
                                                            T* __restrict__ xn, T c1, T c2) {
  constexpr int VW = 16 / (int)sizeof(T);
  constexpr int LR = L * ES;
  static_assert(LR <= 64, "a row's lanes stay inside one wavefront");
  typedef T vec __attribute__((ext_vector_type(VW)));
  const int64_t row = ((int64_t)xcd_block(blockIdx.x, gridDim.x) * kNT + threadIdx.x) / LR;
  if (row >= n) return;  // all LR lanes of a row leave together
  const int sub = threadIdx.x & (LR - 1);
  const int eg = sub / L;
  const int c0 = (sub % L) * VW;
  const bool on = c0 < k;
  vec acc = (vec)(T(0));
  if (on) {
    const int s = rp[row], e = rp[row + 1];
    int q = s + eg;
    for (; q + 3 * ES < e; q += 4 * ES) {
      const int j0 = ci[q], j1 = ci[q + ES], j2 = ci[q + 2 * ES], j3 = ci[q + 3 * ES];
      const T v0 = val[q], v1 = val[q + ES], v2 = val[q + 2 * ES], v3 = val[q + 3 * ES];
      const vec g0 = *(const vec*)(x + (int64_t)j0 * k + c0), g1 = *(const vec*)(x + (int64_t)j1 * k + c0);
      const vec g2 = *(const vec*)(x + (int64_t)j2 * k + c0), g3 = *(const vec*)(x + (int64_t)j3 * k + c0);
      acc += v0 * g0;
      acc += v1 * g1;
      acc += v2 * g2;
      acc += v3 * g3;
    }
    for (; q < e; q += ES) acc += val[q] * *(const vec*)(x + (int64_t)ci[q] * k + c0);
  }
#pragma unroll
  for (int off = LR / 2; off >= L; off >>= 1) {
#pragma unroll
    for (int j = 0; j < VW; ++j) acc[j] += shfl_xor_t(acc[j], off, LR);
  }
  if (!on || eg != 0) return;
  const int64_t idx = row * k + c0;
  if (MODE == kAssign) {
    *(vec*)(y + idx) = acc;
  } else if (MODE == kAssignScale) {
    *(vec*)(y + idx) = acc;
    const vec v = (c1 * (T)dinv[row]) * acc;
    *(vec*)(xn + idx) = v;
    if (d) *(vec*)(d + idx) = v;
  } else if (MODE == kResid) {
    *(vec*)(y + idx) = *(const vec*)(b + idx) - acc;
  } else if (MODE == kAdd) {
    *(vec*)(y + idx) += acc;
  } else if (MODE == kJacobi) {
    *(vec*)(xn + idx) = *(const vec*)(x + idx) + (c1 * dinv[row]) * (*(const vec*)(b + idx) - acc);
  } else {  // kCheb
    const vec r = dinv[row] * (*(const vec*)(b + idx) - acc);
    const vec dn = (c1 != T(0) ? c1 * *(const vec*)(d + idx) : (vec)(T(0))) + c2 * r;
    *(vec*)(d + idx) = dn;
    *(vec*)(xn + idx) = *(const vec*)(x + idx) + dn;
  }
}

// k right-hand sides on the sliced-ELL copy with one lane per row in its
// layout (64-row slices): L lanes per row, each owning VW = 16 / sizeof(T)
// consecutive columns gathered as one 16-byte load; a slice takes L
// wavefronts, each over 64 / L of its rows, so a step reads the 2-byte codes
// and values of those rows as one contiguous run.  Entries in row order,
// padding (value 0) last: the per-column sums are those of
// csr_multi_vec_kernel.
template <typename T, int L, int MODE, int VW = 16 / (int)sizeof(T)>
__global__ void __launch_bounds__(kNT) sell_multi_kernel(int64_t n, int k, int64_t nslices, SellView S,
                                                       const T* __restrict__ sv, const T* __restrict__ x,
                                                       T* __restrict__ y, const T* __restrict__ b,
                                                       const T* __restrict__ dinv, T* __restrict__ d,
                                                       T* __restrict__ xn, T c1, T c2) {
  constexpr int RW = 64 / L;  // rows per wavefront
  typedef T vec __attribute__((ext_vector_type(VW)));
  const int gw = __builtin_amdgcn_readfirstlane((int)(xcd_block(blockIdx.x, gridDim.x) * (kNT / 64) + (threadIdx.x >> 6)));
  const int slice = gw / L;
  if (slice >= nslices) return;
  const int lane = threadIdx.x & 63;
  const int rl = (gw % L) * RW + lane / L;  // row position inside the slice
  const int c0 = (lane % L) * VW;
  const int off = __builtin_amdgcn_readfirstlane(S.sp[slice]);
  const int w = __builtin_amdgcn_readfirstlane((S.sp[slice + 1] - off) >> 6);
  const int32_t* wp = S.swin + slice * kSellWindows;
  const SellWin W{__builtin_amdgcn_readfirstlane(wp[0]), __builtin_amdgcn_readfirstlane(wp[1]),
                  __builtin_amdgcn_readfirstlane(wp[2]), __builtin_amdgcn_readfirstlane(wp[3]),
                  __builtin_amdgcn_readfirstlane(wp[4]), __builtin_amdgcn_readfirstlane(wp[5]),
                  __builtin_amdgcn_readfirstlane(wp[6]), __builtin_amdgcn_readfirstlane(wp[7])};
  const bool on = c0 < k;
  vec acc = (vec)(T(0));
  const T* vp = sv + off + rl;
  if (on) {
    if (W.b0 >= 0) {
      const uint16_t* cp = S.sc16 + off + rl;
      int q = 0;
      for (; q + 4 <= w; q += 4) {
        const int j0 = sell_col(cp[64 * q], W), j1 = sell_col(cp[64 * (q + 1)], W);
        const int j2 = sell_col(cp[64 * (q + 2)], W), j3 = sell_col(cp[64 * (q + 3)], W);
        const T v0 = vp[64 * q], v1 = vp[64 * (q + 1)], v2 = vp[64 * (q + 2)], v3 = vp[64 * (q + 3)];
        const vec g0 = *(const vec*)(x + (int64_t)j0 * k + c0), g1 = *(const vec*)(x + (int64_t)j1 * k + c0);
        const vec g2 = *(const vec*)(x + (int64_t)j2 * k + c0), g3 = *(const vec*)(x + (int64_t)j3 * k + c0);
        acc += v0 * g0;
        acc += v1 * g1;
        acc += v2 * g2;
        acc += v3 * g3;
      }
      for (; q < w; ++q) acc += vp[64 * q] * *(const vec*)(x + (int64_t)sell_col(cp[64 * q], W) * k + c0);
    } else {
      const int32_t* cp = S.sc + off + rl;
      int q = 0;
      for (; q + 4 <= w; q += 4) {
        const int j0 = cp[64 * q], j1 = cp[64 * (q + 1)], j2 = cp[64 * (q + 2)], j3 = cp[64 * (q + 3)];
        const T v0 = vp[64 * q], v1 = vp[64 * (q + 1)], v2 = vp[64 * (q + 2)], v3 = vp[64 * (q + 3)];
        const vec g0 = *(const vec*)(x + (int64_t)j0 * k + c0), g1 = *(const vec*)(x + (int64_t)j1 * k + c0);
        const vec g2 = *(const vec*)(x + (int64_t)j2 * k + c0), g3 = *(const vec*)(x + (int64_t)j3 * k + c0);
        acc += v0 * g0;
        acc += v1 * g1;
        acc += v2 * g2;
        acc += v3 * g3;
      }
      for (; q < w; ++q) acc += vp[64 * q] * *(const vec*)(x + (int64_t)cp[64 * q] * k + c0);
    }
  }
  const int64_t pos = (int64_t)slice * 64 + rl;
  if (!on || pos >= n) return;
  const int64_t row = S.srow ? (int64_t)S.srow[pos] : pos;
  const int64_t idx = row * k + c0;
  if (const T* sd = sell_diag<T>(S)) acc += sd[row] * *(const vec*)(x + idx);  // the diagonal term, last
  if (MODE == kAssign) {
    *(vec*)(y + idx) = acc;
  } else if (MODE == kAssignScale) {
    *(vec*)(y + idx) = acc;
    const vec v = (c1 * (T)dinv[row]) * acc;
    *(vec*)(xn + idx) = v;
    if (d) *(vec*)(d + idx) = v;
  } else if (MODE == kResid) {
    *(vec*)(y + idx) = *(const vec*)(b + idx) - acc;
  } else if (MODE == kAdd) {
    *(vec*)(y + idx) += acc;
  } else if (MODE == kJacobi) {
    *(vec*)(xn + idx) = *(const vec*)(x + idx) + (c1 * dinv[row]) * (*(const vec*)(b + idx) - acc);
  } else {  // kCheb
    const vec r = dinv[row] * (*(const vec*)(b + idx) - acc);
    const vec dn = (c1 != T(0) ? c1 * *(const vec*)(d + idx) : (vec)(T(0))) + c2 * r;
    *(vec*)(d + idx) = dn;
    *(vec*)(xn + idx) = *(const vec*)(x + idx) + dn;
  }
}

// ---- k right-hand sides on the LDS-staged copy ------------------------------------
// A block of L.bs slices takes the columns in chunks of VW * LN: it stages x's
// rows at its distinct columns (one gather of VW * LN values per listed
// column, 3.4 of them per row at 161^3 against 14 entries), then LN lanes per
// row, VW consecutive columns each, read the entries' x rows from LDS.  With x
// gathered per entry the address unit bounded the pass.  What bounds it now is
// the chain list -> columns -> x -> LDS -> row vectors of each block, hidden
// only by other wavefronts: full occupancy (at most 64 registers) beats loads
// issued ahead (161^3, 16 columns, FP32 step 479 us unstaged, 417 staged; 476
// with the row's vectors and entries loaded before the staging at 5 wavefronts
// a SIMD).  A lane takes 16 bytes of columns, so that few lanes load each entry:
// 161^3, 4 columns, FP32 step 161 us by one lane a row, 309 by four lanes of one
// column each, 181 unstaged; FP64 301, 380 and 333.  FP64 rows of 16 columns have eight lanes; there the lanes of a
// quad load one entry each of four and share them by DPP (operator + p.q 738
// us unstaged, 747 staged with all lanes loading every code and value, the
// address unit 70 % busy, 721 shared).  61 x 58 x 73, 5 columns in 8, FP64
// step: 39.8 us with a lane per column on the CSR arrays, 23.2 us.
// Per column the sum is in entry order, as in sell_multi_kernel.  DOT 1:
// per-block, per-column partials of x.y (the operator's p.q); DOT 2: of r.xn
// (the last smoothing step's r.z).
template <typename T, int VW>
struct VecOf {
  typedef T type __attribute__((ext_vector_type(VW)));
};

// v of lane J of each quad
template <int J>
__device__ __forceinline__ int quad_bcast(int v) {
  return __builtin_amdgcn_mov_dpp(v, J * 0x55, 0xf, 0xf, true);
}
template <int J>
__device__ __forceinline__ double quad_bcast(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint64_t lo = (uint32_t)quad_bcast<J>((int)(uint32_t)u), hi = (uint32_t)quad_bcast<J>((int)(uint32_t)(u >> 32));
  return __builtin_bit_cast(double, hi << 32 | lo);
}

// acc += v_j * x row of entry j, j = 0..3 of the quad's four entries (m of them real)
template <typename T, typename Vec>
__device__ __forceinline__ void quad_entries(int c, T v, int m, const Vec* xl, int stride, Vec& acc) {
  acc += quad_bcast<0>(v) * xl[quad_bcast<0>(c) * stride];
  if (m > 1) acc += quad_bcast<1>(v) * xl[quad_bcast<1>(c) * stride];
  if (m > 2) acc += quad_bcast<2>(v) * xl[quad_bcast<2>(c) * stride];
  if (m > 3) acc += quad_bcast<3>(v) * xl[quad_bcast<3>(c) * stride];
}

// the row's sum over its w entries; cp, vp: the row's first code and value,
// xl: this lane's piece of the staged rows
template <typename T, int LN, typename Vec>
__device__ __forceinline__ Vec multi_row_sum(const uint16_t* cp, const T* vp, int w, const Vec* xl) {
  Vec acc = (Vec)(T(0));
  if constexpr (sizeof(T) == 8 && LN >= 4) {
    const int q4 = threadIdx.x & 3;  // entry 4 g + q4 of the row is this lane's of group g
    for (int g = 0; 4 * g < w; ++g) {
      int ec = 0;
      T ev = T(0);
      if (4 * g + q4 < w) {
        ec = cp[64 * (4 * g + q4)];
        ev = vp[64 * (4 * g + q4)];
      }
      quad_entries(ec, ev, w - 4 * g, xl, LN, acc);
    }
  } else {
    int q = 0;
    for (; q + 4 <= w; q += 4) {
      unsigned i[4];
      T v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        i[j] = cp[64 * (q + j)];
        v[j] = vp[64 * (q + j)];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) acc += v[j] * xl[i[j] * LN];
    }
    for (; q < w; ++q) acc += vp[64 * q] * xl[cp[64 * q] * LN];
  }
  return acc;
}

constexpr int kMultiSlices = 2;  // slices per block at most

template <typename T, int VW, int LN, int MODE, int DOT>
__global__ void __launch_bounds__(64 * kMultiSlices * LN, 8) sell_lds_multi_kernel(
    int64_t n, int k, int64_t nslices, SellView S, LdsView L, const T* __restrict__ sv, const T* __restrict__ x,
    T* __restrict__ y, const T* __restrict__ b, const T* __restrict__ dinv, T* __restrict__ d, T* __restrict__ xn,
    T c1, T c2, const double* __restrict__ r64, double* __restrict__ partials) {
  typedef typename VecOf<T, VW>::type vec;
  static_assert(64 % LN == 0, "rows of one slice per wavefront");
  extern __shared__ unsigned char lds_raw[];
  vec* xs = reinterpret_cast<vec*>(lds_raw);
  __shared__ double s_dot[DOT ? kMultiSlices * LN * VW * LN : 1];
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const int tid = threadIdx.x, nt = blockDim.x;
  const int lc0 = L.lcs[blk], npiece = (L.lcs[blk + 1] - lc0) * LN;
  const int rl = tid / LN, piece = tid % LN;
  const int slice = __builtin_amdgcn_readfirstlane((int)blk * L.bs + (rl >> 6));
  const int64_t pos = (int64_t)slice * 64 + (rl & 63);
  const bool on = slice < nslices && pos < n;  // the same for the lanes of a row
  int off = 0, w = 0;
  if (slice < nslices) {
    off = __builtin_amdgcn_readfirstlane(S.sp[slice]);
    w = __builtin_amdgcn_readfirstlane((S.sp[slice + 1] - off) >> 6);
  }
  const T* vp = sv + off + (rl & 63);
  const uint16_t* cp = L.lc + off + (rl & 63);
  int64_t row = pos;
  if (on && S.srow) row = S.srow[pos];
  const T* sdp = sell_diag<T>(S);
  for (int cb = 0; cb < k; cb += VW * LN) {
    if (cb) __syncthreads();  // the previous chunk's LDS rows are read
    for (int t = tid; t < npiece; t += nt) {
      const int c = cb + (t % LN) * VW;
      if (c < k) xs[t] = *(const vec*)(x + (int64_t)L.lcols[lc0 + t / LN] * k + c);
    }
    __syncthreads();
    const int c = cb + piece * VW;
    double part[VW];
#pragma unroll
    for (int j = 0; j < VW; ++j) part[j] = 0.0;
    if (on) {
      vec acc = multi_row_sum<T, LN>(cp, vp, w, xs + piece);
      if (c < k) {
        const int64_t idx = row * k + c;
        vec xv = (vec)(T(0));
        if (sdp || MODE == kJacobi || MODE == kCheb || DOT == 1) xv = *(const vec*)(x + idx);
        if (sdp) acc += sdp[row] * xv;  // the diagonal term, last
        vec out = acc;
        if (MODE == kAssign) {
          *(vec*)(y + idx) = acc;
        } else if (MODE == kAssignScale) {
          *(vec*)(y + idx) = acc;
          out = (c1 * dinv[row]) * acc;
          *(vec*)(xn + idx) = out;
          if (d) *(vec*)(d + idx) = out;
        } else if (MODE == kResid) {
          *(vec*)(y + idx) = *(const vec*)(b + idx) - acc;
        } else if (MODE == kAdd) {
          *(vec*)(y + idx) += acc;
        } else if (MODE == kJacobi) {
          out = xv + (c1 * dinv[row]) * (*(const vec*)(b + idx) - acc);
          *(vec*)(xn + idx) = out;
        } else {  // kCheb (d is not needed after a last step, DOT 2)
          const vec r = dinv[row] * (*(const vec*)(b + idx) - acc);
          const vec dn = (c1 != T(0) ? c1 * *(const vec*)(d + idx) : (vec)(T(0))) + c2 * r;
          if (DOT != 2) *(vec*)(d + idx) = dn;
          out = xv + dn;
          *(vec*)(xn + idx) = out;
        }
        if (DOT == 1) {
#pragma unroll
          for (int j = 0; j < VW; ++j) part[j] = (double)xv[j] * (double)acc[j];
        } else if (DOT == 2) {
#pragma unroll
          for (int j = 0; j < VW; ++j) part[j] = r64[idx + j] * (double)out[j];
        }
      }
    }
    if (DOT) {
      // over the wavefront's rows, then over the wavefronts (fixed order)
#pragma unroll
      for (int j = 0; j < VW; ++j) {
#pragma unroll
        for (int o = 32; o >= LN; o >>= 1) part[j] += __shfl_xor(part[j], o, 64);
        if ((tid & 63) < LN) s_dot[((tid >> 6) * LN + piece) * VW + j] = part[j];
      }
      __syncthreads();
      if (tid < VW * LN && cb + tid < k) {
        double t = 0.0;
        for (int i = 0; i < (nt >> 6); ++i) t += s_dot[i * VW * LN + tid];
        partials[(int64_t)(cb + tid) * gridDim.x + blockIdx.x] = t;
      }
    }
  }
}

// ---- reductions ---------------------------------------------------------------

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Sum of v over the block of 64 * waves threads (fixed order); result valid in
// thread 0.
__device__ __forceinline__ double block_sum(double v, double* s_buf, int waves = kNT / 64) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_buf[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < waves; ++i) r += s_buf[i];
  __syncthreads();
  return r;
}

// Per-column block partials for row-major (n x k) data: thread (row, c) with
// c = tid % KP.  Writes partials[c * gridDim.x + blockIdx.x] for c < k (a
// column's partials are consecutive for the finish).
template <int KP>
__device__ __forceinline__ void block_col_partials(double v, int k, double* s_buf, double* partials) {
  if (KP == 1) {
    double r = block_sum(v, s_buf);
    if (threadIdx.x == 0) partials[blockIdx.x] = r;
    return;
  }
  s_buf[threadIdx.x] = v;
  __syncthreads();
  if ((int)threadIdx.x < k) {
    double s = 0.0;
    for (int j = threadIdx.x; j < kNT; j += KP) s += s_buf[j];
    partials[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = s;
  }
  __syncthreads();
}

}  // namespace fem
