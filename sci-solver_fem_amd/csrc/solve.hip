// V-cycle and preconditioned CG.
//
// Reference path being replaced: CG_Flex_Cycle (src/core/cuda/cgcycle.cu:7-69),
// AMG_Level::cycle / cycle_level0 (src/core/cuda/amg_level.cu:22-128) and the
// smoother kernels of src/core/cuda/gauss_seidel.cu (preRRRFullSymmetric
// :2018-2261, postPCRFullSymmetric :4409-4662).
//
// Differences by design (results are compared on the solution, which the
// preconditioner does not change):
//  * the V-cycle is symmetric (same polynomial smoother before and after the
//    coarse correction), so plain CG is valid for it;
//  * the outer residual stays FP64 and is never overwritten by the V-cycle;
//  * the stop test is re-checked on the true residual b - A x;
//  * scalars (alpha, beta, norms) stay on the device; the host reads one
//    vector of squared residual norms per iteration.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>

#include "fem_internal.hpp"
#include "kernels.hpp"

namespace fem {

namespace {

enum { S_RZ = 0, S_PQ, S_ALPHA, S_BETA, S_RR, S_BB, S_ACT, S_RZN, S_TRUE, S_SEQ, S_COUNT };

// host-mapped record of one |r|^2 finish: act[64], rr[64], sequence number;
// two records (by the parity of the sequence number)
constexpr int kActRec = 136;

int pow2_at_least(int k) {
  int p = 1;
  while (p < k) p <<= 1;
  return p;
}

// lanes per row of the CSR kernels, from the average row length (measured at
// 161^3: 64-entry coarse rows run fastest with 16 lanes, 100-entry
// restriction rows with 32)
int lanes_for(const Csr& A) {
  double avg = A.n ? (double)A.nnz / (double)A.n : 1.0;
  if (avg <= 6) return 4;
  if (avg <= 12) return 8;
  if (avg <= 80) return 16;
  if (avg <= 200) return 32;
  return 64;
}

const Csr& level_A(const Handle& h, int l) { return l == 0 ? h.A : h.H.levels[l]->A; }

template <typename V>
const V* vals_of(const Csr& A);
template <>
const double* vals_of<double>(const Csr& A) { return A.v64.get(); }
template <>
const float* vals_of<float>(const Csr& A) { return A.v32.get(); }

template <typename V>
const V* dinv_of(const Level& L);
template <>
const double* dinv_of<double>(const Level& L) { return L.dinv64.get(); }
template <>
const float* dinv_of<float>(const Level& L) { return L.dinv32.get(); }

template <typename T>
struct LV;
template <>
struct LV<double> {
  static double* x(Level& L) { return L.x64.get(); }
  static double* t(Level& L) { return L.t64.get(); }
  static double* b(Level& L) { return L.b64.get(); }
  static double* r(Level& L) { return L.r64.get(); }
  static double* d(Level& L) { return L.d64.get(); }
};
template <>
struct LV<float> {
  static float* x(Level& L) { return L.x32.get(); }
  static float* t(Level& L) { return L.t32.get(); }
  static float* b(Level& L) { return L.b32.get(); }
  static float* r(Level& L) { return L.r32.get(); }
  static float* d(Level& L) { return L.d32.get(); }
};

template <typename V, typename T, int MODE, int G>
void launch_vec(const Csr& A, const V* val, const T* x, T* y, const T* b, const V* dinv, T* d, T* xn, T c1, T c2,
                hipStream_t s) {
  unsigned grid = grid_for(A.n * G, kNT);
  csr_vec_kernel<V, T, G, MODE><<<grid, kNT, 0, s>>>(A.n, A.rp.get(), A.ci.get(), val, x, y, b, dinv, d, xn, c1, c2);
}

template <typename T, int MODE, int L, int ES>
void launch_multi_split(const Csr& A, int k, const T* val, const T* x, T* y, const T* b, const T* dinv, T* d, T* xn,
                        T c1, T c2, hipStream_t s) {
  unsigned grid = grid_for(A.n * L * ES, kNT);
  csr_multi_split_kernel<T, L, ES, MODE><<<grid, kNT, 0, s>>>(A.n, k, A.rp.get(), A.ci.get(), val, x, y, b, dinv, d,
                                                              xn, c1, c2);
}

// Entry groups per row of the multi-column CSR kernels: enough for at most
// ~16 entries each (coarse operators, restrictions), within one wavefront.
int entry_split(const Csr& A, int L) {
  const double avg = A.n ? (double)A.nnz / (double)A.n : 0.0;
  int es = 1;
  while (es * L < 64 && avg > 16.0 * es) es *= 2;
  return es;
}

template <typename T, int MODE, int L>
void launch_multi_vec(const Csr& A, int k, const T* val, const T* x, T* y, const T* b, const T* dinv, T* d, T* xn,
                      T c1, T c2, hipStream_t s) {
  switch (L < 64 ? entry_split(A, L) : 1) {
    case 1: break;
    case 2: launch_multi_split<T, MODE, L, (L <= 32 ? 2 : 1)>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); return;
    case 4: launch_multi_split<T, MODE, L, (L <= 16 ? 4 : 1)>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); return;
    case 8: launch_multi_split<T, MODE, L, (L <= 8 ? 8 : 1)>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); return;
    case 16: launch_multi_split<T, MODE, L, (L <= 4 ? 16 : 1)>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); return;
    case 32: launch_multi_split<T, MODE, L, (L <= 2 ? 32 : 1)>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); return;
    default: launch_multi_split<T, MODE, L, (L <= 1 ? 64 : 1)>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); return;
  }
  unsigned grid = grid_for(A.n * L, kNT);
  csr_multi_vec_kernel<T, L, MODE><<<grid, kNT, 0, s>>>(A.n, k, A.rp.get(), A.ci.get(), val, x, y, b, dinv, d, xn,
                                                        c1, c2);
}

template <typename T>
const T* svals_of(const Csr& A);
template <>
const double* svals_of<double>(const Csr& A) { return A.s64.get(); }
template <>
const float* svals_of<float>(const Csr& A) { return A.s32.get(); }

template <typename T, int MODE, int G>
void launch_sell(const Csr& A, const T* x, T* y, const T* b, const T* dinv, T* d, T* xn, T c1, T c2, hipStream_t s) {
  sell_kernel<T, MODE, G><<<grid_for(A.nslices, kNT / 64), kNT, 0, s>>>(A.n, A.nslices, sell_view(A), svals_of<T>(A), x,
                                                                       y, b, dinv, d, xn, c1, c2);
}

// columns per lane of the multi-column sliced kernel: 4 (FP32 16-byte, FP64
// 32-byte gathers; measured at 161^3 with 16 columns: FP64 with 2 per lane
// 12 % slower, FP32 with 8 per lane 7 % slower)
template <typename T>
constexpr int sell_multi_cols() { return 4; }
// longer average rows take the entry-split CSR kernel for k columns (161^3
// level 1, ~45 entries per row: 45 us against ~69 us on the sliced copy)
constexpr int64_t kMultiSellRow = 24;

template <typename T, int MODE, int L>
void launch_sell_multi(const Csr& A, int k, const T* x, T* y, const T* b, const T* dinv, T* d, T* xn, T c1, T c2,
                       hipStream_t s) {
  unsigned grid = grid_for(A.nslices * L, kNT / 64);
  sell_multi_kernel<T, L, MODE, sell_multi_cols<T>()><<<grid, kNT, 0, s>>>(A.n, k, A.nslices, sell_view(A),
                                                                           svals_of<T>(A), x, y, b, dinv, d, xn, c1, c2);
}

constexpr int kLdsHead = 16;         // steps
constexpr int64_t kLdsHeadRow = 20;  // average row length above which no head is loaded

// Launch on an LDS-staged copy with values of `vsize` bytes: f(head steps,
// blocks, threads).  Loading the first 16 steps before the staging barrier
// pays where that latency is exposed, at the price of registers (FP32 48,
// FP64 66 per lane).  Measured (Chebyshev step, before -> with the head):
//  * 97^3, blocks of 2 slices: FP32 25.2 -> 20.9 us, FP64 operator + p.q
//    35.8 -> 31.9 us; 49^3 FP64 7.6 -> 6.6 us;
//  * 161^3 FP32, blocks of 8: 88.5 -> 76.6 us (505 MB: 6.6 TB/s); FP16 alike;
//  * FP64 in blocks of 8 fills the memory system anyway and loses a
//    wavefront per SIMD to the registers: 8, 12, 16 head steps give 88.7,
//    93.8, 85.0 us at 131 x 150 x 119 against 81.6 us without, batches of
//    eight 82.0 against 80.4 in fours;
//  * rows longer than the head (161^3 level 1, ~46 entries): 16.9 us without,
//    18.5 with, 15.7 without in batches of eight instead of four; their blocks
//    of 2 slices stage with four wavefronts;
//  * 2D operators (~7 entries per row) need 8 steps: 1003 x 701 FP64 operator
//    + p.q 18.2 -> 13.3 us (15.7 with 16 steps' registers);
//  * fewer blocks than CUs (65^2: 34): a launch is all latency, and the longer
//    code of the head costs more than it hides (3.25 us against 3.6).
template <typename Fn>
void lds_launch(const Csr& A, size_t vsize, Fn&& f) {
  const unsigned nb = (unsigned)((A.nslices + A.lds.bs - 1) / A.lds.bs);
  const unsigned nt = 64u * (unsigned)A.lds.bs;
  const bool lengths = A.srow.size() > 0;  // rows in length order (prolongators)
  if (A.lds.bs > 2 && vsize == 8)
    f(std::integral_constant<int, 0>{}, nb, nt);
  else if (nb < 256u || A.nnz > kLdsHeadRow * A.n)
    f(std::integral_constant<int, kLdsBatch>{}, nb, nt < 256u ? 256u : nt);
  else if (A.nnz <= 8 * A.n && !lengths)
    f(std::integral_constant<int, 8>{}, nb, nt);
  else
    f(std::integral_constant<int, kLdsHead>{}, nb, nt);
}

// ---- several columns on the staged copy
constexpr int kMultiLds = 122880;  // bytes of x rows a block stages at most

const LdsList& multi_list(const Csr& A) { return A.ldm.bs > 0 ? A.ldm : A.lds; }

// columns per lane (16 bytes) and lanes per row: 4, 8 and 16 columns by one,
// two and four lanes in FP32, twice as many in FP64.  Operators
// with a staged copy take it whatever their row length (161^3 level 1, ~46
// entries: 43.9 us a step against 52.2 for the entry-split CSR kernel)
template <typename T>
constexpr int kMultiCols = 16 / (int)sizeof(T);
template <typename T>
int multi_lanes(int k) { return std::min(pow2_at_least(k / kMultiCols<T>), sizeof(T) == 8 ? 8 : 4); }

template <typename T>
size_t multi_lds(const Csr& A, int k) {
  return (size_t)multi_list(A).maxc * kMultiCols<T> * multi_lanes<T>(k) * sizeof(T);
}

template <typename T>
bool multi_staged(const Csr& A, int k) {
  const LdsList& M = multi_list(A);
  return k > 1 && k % kMultiCols<T> == 0 && A.nslices > 0 && A.sell_g == 1 && svals_of<T>(A) && M.bs > 0 &&
         M.bs <= kMultiSlices && multi_lds<T>(A, k) <= (size_t)kMultiLds;
}

unsigned multi_blocks(const Csr& A) { return (unsigned)((A.nslices + multi_list(A).bs - 1) / multi_list(A).bs); }

template <typename T, int MODE, int DOT>
void launch_lds_multi(const Csr& A, int k, const T* x, T* y, const T* b, const T* dinv, T* d, T* xn, T c1, T c2,
                      const double* r64, double* partials, hipStream_t s) {
  const LdsList& M = multi_list(A);
  auto go = [&](auto ln) {
    constexpr int VW = kMultiCols<T>, LN = decltype(ln)::value;
    sell_lds_multi_kernel<T, VW, LN, MODE, DOT><<<multi_blocks(A), 64 * M.bs * LN, multi_lds<T>(A, k), s>>>(
        A.n, k, A.nslices, sell_view(A), lds_view(M), svals_of<T>(A), x, y, b, dinv, d, xn, c1, c2, r64, partials);
  };
  switch (multi_lanes<T>(k)) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    default:
      if constexpr (sizeof(T) == 8) go(std::integral_constant<int, 8>{});
      break;
  }
}

// y/xn = f(A x) for k right-hand sides; MODE selects the epilogue.  One RHS
// uses the sliced-ELL copy when it exists, otherwise CSR with G lanes per row.
template <typename T, int MODE>
void spmv_op(const Csr& A, int k, const T* x, T* y, const T* b, const T* dinv, T* d, T* xn, T c1, T c2,
             hipStream_t s) {
  if (A.n == 0) return;
  const T* val = vals_of<T>(A);
  if (k == 1 && A.nslices > 0 && svals_of<T>(A) && A.lds.bs > 0) {
    lds_launch(A, sizeof(T), [&](auto head, unsigned nb, unsigned nt) {
      sell_lds_kernel<T, MODE, head.value><<<nb, nt, sizeof(T) * (size_t)A.lds.maxc, s>>>(
          A.n, A.nslices, sell_view(A), lds_view(A.lds), svals_of<T>(A), x, y, b, dinv, d, xn, c1, c2);
    });
  } else if (k == 1 && A.nslices > 0 && svals_of<T>(A)) {
    switch (A.sell_g) {
      case 1: launch_sell<T, MODE, 1>(A, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 2: launch_sell<T, MODE, 2>(A, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 4: launch_sell<T, MODE, 4>(A, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 8: launch_sell<T, MODE, 8>(A, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 16: launch_sell<T, MODE, 16>(A, x, y, b, dinv, d, xn, c1, c2, s); break;
      default: launch_sell<T, MODE, 32>(A, x, y, b, dinv, d, xn, c1, c2, s); break;
    }
  } else if (k == 1) {
    switch (lanes_for(A)) {
      case 4: launch_vec<T, T, MODE, 4>(A, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 8: launch_vec<T, T, MODE, 8>(A, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 16: launch_vec<T, T, MODE, 16>(A, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 32: launch_vec<T, T, MODE, 32>(A, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      default: launch_vec<T, T, MODE, 64>(A, val, x, y, b, dinv, d, xn, c1, c2, s); break;
    }
  } else if (MODE != kAdd && multi_staged<T>(A, k)) {  // prolongators: short rows, 196 us unstaged, 202 staged
    launch_lds_multi<T, MODE, 0>(A, k, x, y, b, dinv, d, xn, c1, c2, nullptr, nullptr, s);
  } else if (k % sell_multi_cols<T>() == 0 && A.nslices > 0 && A.sell_g == 1 && svals_of<T>(A) &&
             A.nnz <= kMultiSellRow * A.n) {
    // column groups on the sliced-ELL copy
    switch (pow2_at_least(k / sell_multi_cols<T>())) {
      case 1: launch_sell_multi<T, MODE, 1>(A, k, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 2: launch_sell_multi<T, MODE, 2>(A, k, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 4: launch_sell_multi<T, MODE, 4>(A, k, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 8: launch_sell_multi<T, MODE, 8>(A, k, x, y, b, dinv, d, xn, c1, c2, s); break;
      default: launch_sell_multi<T, MODE, 16>(A, k, x, y, b, dinv, d, xn, c1, c2, s); break;
    }
  } else {
    // 16-byte column groups (all multi-column vectors here come from hipMalloc;
    // padded_columns keeps k a multiple of the group)
    if (k % (16 / (int)sizeof(T)) != 0) fail(FEM_ERR_STATE, "column count is not padded");
    switch (pow2_at_least(k / (16 / (int)sizeof(T)))) {
      case 1: launch_multi_vec<T, MODE, 1>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 2: launch_multi_vec<T, MODE, 2>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 4: launch_multi_vec<T, MODE, 4>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 8: launch_multi_vec<T, MODE, 8>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      case 16: launch_multi_vec<T, MODE, 16>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); break;
      default: launch_multi_vec<T, MODE, 32>(A, k, val, x, y, b, dinv, d, xn, c1, c2, s); break;
    }
  }
  HIP_LAUNCH_CHECK();
}

// ---- elementwise kernels ------------------------------------------------------

// x = c1 * dinv * b (first smoothing step from a zero guess); d = x if d != null
template <typename V, typename Tb, typename T>
__global__ void scale_dinv_kernel(int64_t n, int k, const V* __restrict__ dinv, const Tb* __restrict__ b,
                                  T* __restrict__ x, T* __restrict__ d, T c1) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * k) return;
  int64_t i = t / k;
  T v = c1 * (T)dinv[i] * (T)b[t];
  x[t] = v;
  if (d) d[t] = v;
}

// First level-0 smoothing step of a mixed-precision V-cycle, from the FP64
// Krylov residual: b = fl32(r); x = c1 * dinv * b; d = x if d != null.
__global__ void scale_in_kernel(int64_t n, const float* __restrict__ dinv, const double* __restrict__ r,
                                float* __restrict__ b, float* __restrict__ x, float* __restrict__ d, float c1) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float bv = (float)r[i];
  b[i] = bv;
  const float v = c1 * dinv[i] * bv;
  x[i] = v;
  if (d) d[i] = v;
}

// Last level-0 smoothing step of a mixed-precision V-cycle (one column,
// sliced ELL): the smoothed value goes straight to the FP64 output z, with
// per-block partials of r.z for the PCG beta (d is not needed afterwards).
template <int MODE>
__global__ void __launch_bounds__(kNT) sell_smooth_out_kernel(int64_t n, int64_t nslices, SellView S,
                                                            const float* __restrict__ sv, const float* __restrict__ x,
                                                            const float* __restrict__ b, const float* __restrict__ dinv,
                                                            const float* __restrict__ d, float c1, float c2,
                                                            const double* __restrict__ r, double* __restrict__ z,
                                                            double* __restrict__ partials) {
  __shared__ double s_buf[kNT];
  const int slice =
      __builtin_amdgcn_readfirstlane((int)(xcd_block(blockIdx.x, gridDim.x) * (kNT / 64) + (threadIdx.x >> 6)));
  const int lane = threadIdx.x & 63;
  double part = 0.0;
  if (slice < nslices) {
    float acc = sell_row_sum<float>(S, slice, lane, sv, x);
    const int64_t row = (int64_t)slice * 64 + lane;
    if (row < n) {
      if (S.sd32) acc += S.sd32[row] * x[row];  // the diagonal term, last
      float xn;
      if (MODE == kJacobi) {
        xn = x[row] + c1 * dinv[row] * (b[row] - acc);
      } else {
        const float rr = ntload(dinv + row) * (ntload(b + row) - acc);
        const float dn = (c1 != 0.0f ? c1 * ntload(d + row) : 0.0f) + c2 * rr;
        xn = x[row] + dn;
      }
      const double zv = (double)xn;
      z[row] = zv;
      part = r[row] * zv;
    }
  }
  const double tot = block_sum(part, s_buf);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// The same on the LDS-staged copy: a block per L.bs slices (a wavefront each),
// r.z partials per block.
template <int MODE, int HEAD>
__global__ void __launch_bounds__(kLdsMaxNT) sell_lds_out_kernel(
    int64_t n, int64_t nslices, SellView S, LdsView L, const float* __restrict__ sv, const float* __restrict__ x,
    const float* __restrict__ b, const float* __restrict__ dinv, const float* __restrict__ d, float c1, float c2,
    const double* __restrict__ r, double* __restrict__ z, double* __restrict__ partials) {
  extern __shared__ unsigned char lds_raw[];
  float* xs = reinterpret_cast<float*>(lds_raw);
  __shared__ double s_buf[kLdsMaxNT / 64];
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const LdsWave w = lds_wave(L, blk, n, nslices);
  const int64_t row = w.pos;
  SliceHead<float, HEAD> H;
  float xv = 0.0f, bv = 0.0f, iv = 0.0f, dv = 0.0f, sdv = 0.0f;
  double rv = 0.0;
  LdsStage G;
  G.begin(L, blk);
  if (w.live) lds_head(H, S, L, w.slice, w.lane, sv);
  if (w.on) {
    xv = x[row];
    bv = ntload(b + row);
    iv = ntload(dinv + row);
    if (MODE == kCheb && c1 != 0.0f) dv = ntload(d + row);
    if (S.sd32) sdv = S.sd32[row];
    rv = r[row];
  }
  G.finish<float>(L, x, xs);
  double part = 0.0;
  float acc = w.on ? lds_row_sum<float>(H, L, w.lane, sv, xs) : float(0);
  if (w.on) {
    if (S.sd32) acc += sdv * xv;  // the diagonal term, last
    float xn;
    if (MODE == kJacobi) {
      xn = xv + c1 * iv * (bv - acc);
    } else {
      const float rr = iv * (bv - acc);
      const float dn = (c1 != 0.0f ? c1 * dv : 0.0f) + c2 * rr;
      xn = xv + dn;
    }
    const double zv = (double)xn;
    z[row] = zv;
    part = rv * zv;
  }
  const double tot = block_sum(part, s_buf, blockDim.x >> 6);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// Last level-0 smoothing step of an FP64 V-cycle (one column, staged copy):
// as sell_lds_kernel, with per-block partials of b.xn = r.z for the PCG beta and
// without the write of d.  A dot product of its own is one more launch and
// reads r and z again: 49^3 7.2 + 3.9 us for the two, 7.4 here; 65^2 3.9 + 2.9
// and 4.3 (solves, with the first step in the update: 49^3 3.49 -> 3.36 ms,
// 65^2 1.86 -> 1.77, 12^3 1.31 -> 1.24, 131 x 150 x 119 30.9 -> 30.5).
template <int MODE, int HEAD>
__global__ void __launch_bounds__(kLdsMaxNT) sell_lds_rz_kernel(
    int64_t n, int64_t nslices, SellView S, LdsView L, const double* __restrict__ sv, const double* __restrict__ x,
    const double* __restrict__ b, const double* __restrict__ dinv, double* __restrict__ d, double* __restrict__ xn,
    double c1, double c2, double* __restrict__ partials) {
  extern __shared__ unsigned char lds_raw[];
  double* xs = reinterpret_cast<double*>(lds_raw);
  __shared__ double s_buf[kLdsMaxNT / 64];
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const LdsWave w = lds_wave(L, blk, n, nslices);
  LdsStage G;
  SliceHead<double, HEAD> H;
  SpmvRow<double> R;
  G.begin(L, blk);
  if (w.live) lds_head(H, S, L, w.slice, w.lane, sv);
  if (w.on) R.template load<MODE>(w.pos, S.sd64, x, nullptr, b, dinv, d, c1);
  G.finish<double>(L, x, xs);
  double part = 0.0;
  if (w.on) {
    double acc = lds_row_sum<double>(H, L, w.lane, sv, xs);
    if (S.sd64) acc += R.sd * R.x;  // the diagonal term, last
    part = R.b * R.template store<MODE, true>(w.pos, acc, nullptr, nullptr, xn, c1, c2);
  }
  const double tot = block_sum(part, s_buf, blockDim.x >> 6);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// ---- precision 2: level-0 smoothing in y = D^1/2 x on D^-1/2 A D^-1/2 with
// FP16 off-diagonals (diagonal 1 + eps_i held apart in FP32)

// first step from y = 0: b^ = s fl32(r), y = c1 b^ (d = y if d != null)
__global__ void scale_in_half_kernel(int64_t n, const float* __restrict__ sd, const double* __restrict__ r,
                                     float* __restrict__ bh, float* __restrict__ y, float* __restrict__ d, float c1) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float bv = sd[i] * (float)r[i];
  bh[i] = bv;
  const float v = c1 * bv;
  y[i] = v;
  if (d) d[i] = v;
}

// r^ = b^ - (diag_i y_i + sum_j h_ij y_j); MODE kResid: out = r^;
// kJacobi: yn = y + c1 r^; kCheb: d = c1 d + c2 r^, yn = y + d
template <int MODE>
__global__ void __launch_bounds__(kNT) sell_half_kernel(int64_t n, int64_t nslices, SellView S,
                                                      const uint16_t* __restrict__ sh, const float* __restrict__ diag,
                                                      const float* __restrict__ y, const float* __restrict__ bh,
                                                      float* __restrict__ out, float* __restrict__ d,
                                                      float* __restrict__ yn, float c1, float c2) {
  const int slice =
      __builtin_amdgcn_readfirstlane((int)(xcd_block(blockIdx.x, gridDim.x) * (kNT / 64) + (threadIdx.x >> 6)));
  const int lane = threadIdx.x & 63;
  if (slice >= nslices) return;
  const float acc = sell_row_sum<float, uint16_t>(S, slice, lane, sh, y);
  const int64_t row = (int64_t)slice * 64 + lane;
  if (row >= n) return;
  const float yi = y[row];
  const float r = ntload(bh + row) - (ntload(diag + row) * yi + acc);
  if (MODE == kResid) {
    out[row] = r;
  } else if (MODE == kJacobi) {
    yn[row] = yi + c1 * r;
  } else {
    const float dn = (c1 != 0.0f ? c1 * ntload(d + row) : 0.0f) + c2 * r;
    d[row] = dn;
    yn[row] = yi + dn;
  }
}

// last post-smoothing step: z = s y_new in FP64 and per-block partials of r.z
template <int MODE>
__global__ void __launch_bounds__(kNT) sell_half_out_kernel(int64_t n, int64_t nslices, SellView S,
                                                          const uint16_t* __restrict__ sh,
                                                          const float* __restrict__ diag, const float* __restrict__ sd,
                                                          const float* __restrict__ y, const float* __restrict__ bh,
                                                          const float* __restrict__ d, float c1, float c2,
                                                          const double* __restrict__ r64, double* __restrict__ z,
                                                          double* __restrict__ partials) {
  __shared__ double s_buf[kNT];
  const int slice =
      __builtin_amdgcn_readfirstlane((int)(xcd_block(blockIdx.x, gridDim.x) * (kNT / 64) + (threadIdx.x >> 6)));
  const int lane = threadIdx.x & 63;
  double part = 0.0;
  if (slice < nslices) {
    const float acc = sell_row_sum<float, uint16_t>(S, slice, lane, sh, y);
    const int64_t row = (int64_t)slice * 64 + lane;
    if (row < n) {
      const float yi = y[row];
      const float r = ntload(bh + row) - (ntload(diag + row) * yi + acc);
      float yv;
      if (MODE == kJacobi) {
        yv = yi + c1 * r;
      } else {
        const float dn = (c1 != 0.0f ? c1 * ntload(d + row) : 0.0f) + c2 * r;
        yv = yi + dn;
      }
      const double zv = (double)(sd[row] * yv);
      z[row] = zv;
      part = r64[row] * zv;
    }
  }
  const double tot = block_sum(part, s_buf);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// The same two kernels on the LDS-staged copy: a block of a wavefront per
// slice stages y at its slices' distinct columns once, and every entry reads
// y from LDS through its 16-bit index (same entries in the same order, so the
// same sums).
template <int MODE, int HEAD>
__global__ void __launch_bounds__(kLdsMaxNT) sell_half_lds_kernel(
    int64_t n, int64_t nslices, SellView S, LdsView L, const uint16_t* __restrict__ sh, const float* __restrict__ diag,
    const float* __restrict__ y, const float* __restrict__ bh, float* __restrict__ out, float* __restrict__ d,
    float* __restrict__ yn, float c1, float c2) {
  extern __shared__ unsigned char lds_raw[];
  float* ys = reinterpret_cast<float*>(lds_raw);
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const LdsWave w = lds_wave(L, blk, n, nslices);
  const int64_t row = w.pos;
  SliceHead<uint16_t, HEAD> H;
  float yi = 0.0f, bv = 0.0f, gv = 0.0f, dv = 0.0f;
  LdsStage G;
  G.begin(L, blk);
  if (w.live) lds_head(H, S, L, w.slice, w.lane, sh);
  if (w.on) {
    yi = y[row];
    bv = ntload(bh + row);
    gv = ntload(diag + row);
    if (MODE == kCheb && c1 != 0.0f) dv = ntload(d + row);
  }
  G.finish<float>(L, y, ys);
  float acc = w.on ? lds_row_sum<float>(H, L, w.lane, sh, ys) : float(0);
  if (!w.on) return;
  const float r = bv - (gv * yi + acc);
  if (MODE == kResid) {
    out[row] = r;
  } else if (MODE == kJacobi) {
    yn[row] = yi + c1 * r;
  } else {
    const float dn = (c1 != 0.0f ? c1 * dv : 0.0f) + c2 * r;
    d[row] = dn;
    yn[row] = yi + dn;
  }
}

template <int MODE, int HEAD>
__global__ void __launch_bounds__(kLdsMaxNT) sell_half_lds_out_kernel(
    int64_t n, int64_t nslices, SellView S, LdsView L, const uint16_t* __restrict__ sh, const float* __restrict__ diag,
    const float* __restrict__ sd, const float* __restrict__ y, const float* __restrict__ bh,
    const float* __restrict__ d, float c1, float c2, const double* __restrict__ r64, double* __restrict__ z,
    double* __restrict__ partials) {
  extern __shared__ unsigned char lds_raw[];
  float* ys = reinterpret_cast<float*>(lds_raw);
  __shared__ double s_buf[kLdsMaxNT / 64];
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const LdsWave w = lds_wave(L, blk, n, nslices);
  const int64_t row = w.pos;
  SliceHead<uint16_t, HEAD> H;
  float yi = 0.0f, bv = 0.0f, gv = 0.0f, dv = 0.0f, sv = 0.0f;
  double rv = 0.0;
  LdsStage G;
  G.begin(L, blk);
  if (w.live) lds_head(H, S, L, w.slice, w.lane, sh);
  if (w.on) {
    yi = y[row];
    bv = ntload(bh + row);
    gv = ntload(diag + row);
    if (MODE == kCheb && c1 != 0.0f) dv = ntload(d + row);
    sv = sd[row];
    rv = r64[row];
  }
  G.finish<float>(L, y, ys);
  double part = 0.0;
  float acc = w.on ? lds_row_sum<float>(H, L, w.lane, sh, ys) : float(0);
  if (w.on) {
    const float r = bv - (gv * yi + acc);
    float yv;
    if (MODE == kJacobi) {
      yv = yi + c1 * r;
    } else {
      const float dn = (c1 != 0.0f ? c1 * dv : 0.0f) + c2 * r;
      yv = yi + dn;
    }
    const double zv = (double)(sv * yv);
    z[row] = zv;
    part = rv * zv;
  }
  const double tot = block_sum(part, s_buf, blockDim.x >> 6);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

template <typename Tin, typename Tout>
__global__ void convert_kernel(int64_t m, const Tin* __restrict__ a, Tout* __restrict__ b) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < m) b[t] = (Tout)a[t];
}

// dense coarse solve x = C b with the FP64 inverse C (row-major nc x nc) in
// every precision: b is widened to FP64, the products are summed in FP64 and
// only the result is rounded to the level's vector type; one wave per row
template <typename T>
__global__ void __launch_bounds__(64) coarse_kernel(int64_t nc, int k, const double* __restrict__ C,
                                                   const T* __restrict__ b, T* __restrict__ x) {
  const int64_t i = blockIdx.x;
  const int lane = threadIdx.x;
  for (int c = 0; c < k; ++c) {
    double acc = 0.0;
    for (int64_t j = lane; j < nc; j += 64) acc += C[i * nc + j] * (double)b[j * k + c];
    acc = wave_sum(acc);
    if (lane == 0) x[i * k + c] = (T)acc;
  }
}

// ---- PCG vector kernels (FP64, k columns, row-major) --------------------------
// Each reduction kernel writes one partial per block and column; a one-block
// finish kernel sums them in a fixed order and updates the device scalars.
// (A last-block-done pattern inside the producer would need an agent-scope
// release fence per block, which writes back the XCD's L2 on gfx950.)

// q = A p and per-block partials of p.q (one column)
template <int G>
__global__ void __launch_bounds__(kNT) pcg_spmv_dot_kernel(int64_t n, const int32_t* __restrict__ rp,
                                                         const int32_t* __restrict__ ci, const double* __restrict__ val,
                                                         const double* __restrict__ p, double* __restrict__ q,
                                                         double* __restrict__ partials) {
  __shared__ double s_buf[kNT];
  double part = 0.0;
  const int lane = threadIdx.x & (G - 1);
  // kNT / G rows per pass, one front per XCD
  const XcdRows R = xcd_rows(n, kNT / G);
  for (int64_t row = R.first + threadIdx.x / G; row < R.hi; row += R.step) {
    const int s = rp[row], e = rp[row + 1];
    double acc = 0.0;
    for (int j = s + lane; j < e; j += G) acc += ntload(val + j) * p[ntload(ci + j)];
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, G);
    if (lane == 0) {
      q[row] = acc;
      part += acc * p[row];
    }
  }
  double tot = block_sum(part, s_buf);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// q = A p on the sliced-ELL copy and per-block partials of p.q (one column);
// a wavefront per slice as in the smoother kernels (no grid-stride loop).
__global__ void __launch_bounds__(kNT) pcg_sell_dot_kernel(int64_t n, int64_t nslices, SellView S,
                                                         const double* __restrict__ sv, const double* __restrict__ p,
                                                         double* __restrict__ q, double* __restrict__ partials) {
  __shared__ double s_buf[kNT];
  const int lane = threadIdx.x & 63;
  const int slice =
      __builtin_amdgcn_readfirstlane((int)(xcd_block(blockIdx.x, gridDim.x) * (kNT / 64) + (threadIdx.x >> 6)));
  double part = 0.0;
  if (slice < nslices) {
    double acc = sell_row_sum<double>(S, slice, lane, sv, p);
    const int64_t row = (int64_t)slice * 64 + lane;
    if (row < n) {
      if (S.sd64) acc += S.sd64[row] * p[row];  // the diagonal term, last
      q[row] = acc;
      part = acc * p[row];
    }
  }
  double tot = block_sum(part, s_buf);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// The same on the LDS-staged copy: a block per L.bs slices (a wavefront each),
// p.q partials per block.
template <int HEAD>
__global__ void __launch_bounds__(kLdsMaxNT) pcg_sell_lds_dot_kernel(
    int64_t n, int64_t nslices, SellView S, LdsView L, const double* __restrict__ sv, const double* __restrict__ p,
    double* __restrict__ q, double* __restrict__ partials) {
  extern __shared__ unsigned char lds_raw[];
  double* xs = reinterpret_cast<double*>(lds_raw);
  __shared__ double s_buf[kLdsMaxNT / 64];
  const unsigned blk = xcd_block(blockIdx.x, gridDim.x);
  const LdsWave w = lds_wave(L, blk, n, nslices);
  const int64_t row = w.pos;
  SliceHead<double, HEAD> H;
  double pv = 0.0, sdv = 0.0;
  LdsStage G;
  G.begin(L, blk);
  if (w.live) lds_head(H, S, L, w.slice, w.lane, sv);
  if (w.on) {
    pv = p[row];
    if (S.sd64) sdv = S.sd64[row];
  }
  G.finish<double>(L, p, xs);
  double part = 0.0;
  double acc = w.on ? lds_row_sum<double>(H, L, w.lane, sv, xs) : double(0);
  if (w.on) {
    if (S.sd64) acc += sdv * pv;  // the diagonal term, last
    q[row] = acc;
    part = acc * pv;
  }
  const double tot = block_sum(part, s_buf, blockDim.x >> 6);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// Total of nb <= kFoldParts partials in every thread of the block, the same in
// every block: a kernel that reads alpha or beta sums the partials itself
// instead of waiting for a finish launch (one column, at most kFoldRows rows:
// more blocks would read more partials each).  Two finish
// launches an iteration less: 65^2 1.73 -> 1.69 ms a solve, 12^3 1.23 -> 1.16,
// 49^3 FP64 3.04 -> 3.00, 20^3 1.88 -> 1.84, 300 x 280 mixed 4.33 -> 4.25.
constexpr int kFoldParts = 1024;
constexpr int64_t kFoldRows = 131072;
__device__ __forceinline__ double fold_sum(const double* __restrict__ part, int nb, double* s_buf) {
  __shared__ double s_tot;
  double v = 0.0;
#pragma unroll
  for (int j = 0; j < kFoldParts / kNT; ++j) {
    const int b = (int)threadIdx.x + j * kNT;
    if (b < nb) v += part[b];
  }
  v = block_sum(v, s_buf);
  if (threadIdx.x == 0) s_tot = v;
  __syncthreads();
  return s_tot;
}

// x += alpha p; r -= alpha q; partials of r.r
// (FOLD: one column, alpha from the npq partials of p.q and r.z in slot rz)
// (and bt = fl(r), the FP32 V-cycle's right-hand side, when bt is given; with
// x0 the level-0 smoother's first step from zero on it, or on r itself in an
// FP64 V-cycle: at 131 x 150 x 119 18.6 us and 15.4 us for that step by itself,
// 29.7 us together; 65^2 2.9 and 2.1 us, 3.0 together)
template <int KP, typename T, bool FOLD>
__global__ void __launch_bounds__(kNT) pcg_update_kernel(int64_t n, int k, double* __restrict__ x,
                                                       double* __restrict__ r, const double* __restrict__ p,
                                                       const double* __restrict__ q, double* __restrict__ partials,
                                                       const double* scal, T* __restrict__ bt,
                                                       const T* __restrict__ dinv, T* __restrict__ x0,
                                                       T* __restrict__ d0, T c0, const double* __restrict__ pq,
                                                       int npq, int rz, double* __restrict__ scal_out) {
  __shared__ double s_buf[kNT];
  double alpha = 0.0;
  if (FOLD) {
    const double v = fold_sum(pq, npq, s_buf);
    alpha = (scal[S_ACT] != 0.0 && v != 0.0) ? scal[rz] / v : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      scal_out[S_PQ] = v;
      scal_out[S_ALPHA] = alpha;
    }
  }
  double part = 0.0;
  const int c = threadIdx.x & (KP - 1);
  const int64_t rows_per_grid = (int64_t)gridDim.x * (kNT / KP);
  if (c < k) {
    const double a = FOLD ? alpha : scal[S_ALPHA * k + c];
    for (int64_t row = ((int64_t)blockIdx.x * kNT + threadIdx.x) / KP; row < n; row += rows_per_grid) {
      int64_t t = row * k + c;
      x[t] += a * p[t];
      double rv = r[t] - a * q[t];
      r[t] = rv;
      if (bt) bt[t] = (T)rv;
      if (x0) {  // the level-0 smoother's first step from zero
        const T v = c0 * dinv[row] * (T)rv;
        x0[t] = v;
        if (d0) d0[t] = v;
      }
      part += rv * rv;
    }
  }
  block_col_partials<KP>(part, k, s_buf, partials);
}

// q = A p and per-block, per-column partials of p.q for an even k (operators
// without a staged copy): L lanes per row, two columns per lane as one
// 16-byte load.
template <int L>
__global__ void __launch_bounds__(kNT) pcg_spmm_dot_vec_kernel(int64_t n, int k, const int32_t* __restrict__ rp,
                                                             const int32_t* __restrict__ ci,
                                                             const double* __restrict__ val,
                                                             const double* __restrict__ p, double* __restrict__ q,
                                                             double* __restrict__ partials) {
  typedef double vec __attribute__((ext_vector_type(2)));
  __shared__ double s_buf[2 * kNT];
  const int c0 = (int)(threadIdx.x & (L - 1)) * 2;
  const XcdRows R = xcd_rows(n, kNT / L);
  vec part = (vec)(0.0);
  if (c0 < k) {
    for (int64_t row = R.first + threadIdx.x / L; row < R.hi; row += R.step) {
      const int s = rp[row], e = rp[row + 1];
      vec acc = (vec)(0.0);
      int j = s;
      for (; j + 4 <= e; j += 4) {
        const vec g0 = *(const vec*)(p + (int64_t)ci[j] * k + c0), g1 = *(const vec*)(p + (int64_t)ci[j + 1] * k + c0);
        const vec g2 = *(const vec*)(p + (int64_t)ci[j + 2] * k + c0),
                  g3 = *(const vec*)(p + (int64_t)ci[j + 3] * k + c0);
        acc += val[j] * g0;
        acc += val[j + 1] * g1;
        acc += val[j + 2] * g2;
        acc += val[j + 3] * g3;
      }
      for (; j < e; ++j) acc += val[j] * *(const vec*)(p + (int64_t)ci[j] * k + c0);
      *(vec*)(q + row * k + c0) = acc;
      part += acc * *(const vec*)(p + row * k + c0);
    }
  }
  s_buf[2 * threadIdx.x] = part.x;
  s_buf[2 * threadIdx.x + 1] = part.y;
  __syncthreads();
  if ((int)threadIdx.x < k) {
    const int c = threadIdx.x;
    double sum = 0.0;
    for (int t = c / 2; t < kNT; t += L) sum += s_buf[2 * t + (c & 1)];
    partials[(int64_t)c * gridDim.x + blockIdx.x] = sum;
  }
}

// partials of a.b per column
template <int KP, typename B>
__global__ void __launch_bounds__(kNT) pcg_dot_kernel(int64_t n, int k, const double* __restrict__ a,
                                                    const B* __restrict__ b, double* __restrict__ partials) {
  __shared__ double s_buf[kNT];
  double part = 0.0;
  const int c = threadIdx.x & (KP - 1);
  const int64_t rows_per_grid = (int64_t)gridDim.x * (kNT / KP);
  if (c < k)
    for (int64_t row = ((int64_t)blockIdx.x * kNT + threadIdx.x) / KP; row < n; row += rows_per_grid)
      part += a[row * k + c] * (double)b[row * k + c];
  block_col_partials<KP>(part, k, s_buf, partials);
}

enum FinishMode { F_STORE = 0, F_ALPHA = 1, F_RR = 2, F_BETA = 3, F_FLEX = 4 };

// one block per column: the total of its nb partials, then the scalar update
// 1024 threads so that ~16k partials take a few rounds of independent loads.
// (One block walking all columns took 40 us for 16.)
constexpr int kFinNT = 1024;

__global__ void __launch_bounds__(kFinNT) pcg_finish_kernel(int nb, int k, const double* __restrict__ partials,
                                                          double* __restrict__ scal, int mode, int slot, double tol2,
                                                          double* __restrict__ host_act) {
  __shared__ double s_buf[kFinNT / 64];
  const int c = blockIdx.x;
  const double* __restrict__ part = partials + (int64_t)c * nb;
  double v = 0.0;
#pragma unroll 8
  for (int b = threadIdx.x; b < nb; b += kFinNT) v += part[b];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) s_buf[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x != 0) return;
  v = 0.0;
  for (int w = 0; w < kFinNT / 64; ++w) v += s_buf[w];
  if (mode == F_STORE) {
    scal[slot * k + c] = v;
  } else if (mode == F_ALPHA) {
    scal[S_PQ * k + c] = v;
    scal[S_ALPHA * k + c] = (scal[S_ACT * k + c] != 0.0 && v != 0.0) ? scal[slot * k + c] / v : 0.0;
  } else if (mode == F_RR) {
    if (slot != S_RZ) scal[S_RZ * k + c] = scal[slot * k + c];  // stored there by pcg_p_kernel
    // |r|^2 finishes are numbered on the device (every column counts its
    // own); record n goes to host record n % 2
    const double seq = scal[S_SEQ * k + c] + 1.0;
    scal[S_SEQ * k + c] = seq;
    scal[S_RR * k + c] = v;
    const bool act = scal[S_ACT * k + c] != 0.0 && v > tol2 * scal[S_BB * k + c];
    scal[S_ACT * k + c] = act ? 1.0 : 0.0;
    if (host_act) {
      double* rec = host_act + ((int64_t)seq & 1) * kActRec;
      rec[c] = act ? 1.0 : 0.0;
      rec[64 + c] = v;
      if (c == 0) rec[128] = seq;  // read by the host after this kernel completed
    }
  } else if (mode == F_FLEX) {
    // v = z.q with q = A p of the last step: z.r_old = z.r + alpha z.q, so
    // the flexible (Polak-Ribiere) beta = (z.r - z.r_old) / rz_old =
    // -alpha z.q / rz_old; z.r was stored in S_RZN
    const double rz = scal[S_RZ * k + c];
    scal[S_BETA * k + c] = (scal[S_ACT * k + c] != 0.0 && rz != 0.0) ? -scal[S_ALPHA * k + c] * v / rz : 0.0;
    scal[S_RZ * k + c] = scal[S_RZN * k + c];
  } else {
    const double rz = scal[S_RZ * k + c];
    scal[S_BETA * k + c] = (scal[S_ACT * k + c] != 0.0 && rz != 0.0) ? v / rz : 0.0;
    scal[S_RZ * k + c] = v;
  }
}

// p = z + beta p (z as the preconditioner left it: FP64, or the FP32 V-cycle
// result, converted exactly)
template <typename Z>
__global__ void pcg_p_kernel(int64_t m, int k, const Z* __restrict__ z, double* __restrict__ p,
                             const double* __restrict__ scal) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m) return;
  int c = (int)(t % k);
  p[t] = (double)z[t] + scal[S_BETA * k + c] * p[t];
}

// The same for one column with beta from the nrz partials of r.z; r.z goes to
// S_RZN (other blocks still read S_RZ), moved by the next |r|^2 finish.
template <typename Z>
__global__ void __launch_bounds__(kNT) pcg_p_fold_kernel(int64_t n, const Z* __restrict__ z, double* __restrict__ p,
                                                       double* scal, const double* __restrict__ parts, int nrz) {
  __shared__ double s_buf[kNT];
  const int64_t t = (int64_t)blockIdx.x * kNT + threadIdx.x;
  double zv = 0.0, pv = 0.0;
  if (t < n) {
    zv = (double)z[t];
    pv = p[t];
  }
  const double v = fold_sum(parts, nrz, s_buf);
  const double rz = scal[S_RZ];
  const double beta = (scal[S_ACT] != 0.0 && rz != 0.0) ? v / rz : 0.0;
  if (t == 0) {
    scal[S_RZN] = v;
    scal[S_BETA] = beta;
  }
  if (t < n) p[t] = zv + beta * pv;
}

// x[:, c] = 0 for every column c whose bit is set in mask (k <= 64 columns)
__global__ void zero_cols_kernel(int64_t m, int k, unsigned long long mask, double* __restrict__ x) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < m && ((mask >> (t % k)) & 1ull)) x[t] = 0.0;
}

__global__ void copy_kernel(int64_t m, const double* __restrict__ a, double* __restrict__ b) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < m) b[t] = a[t];
}

unsigned vec_grid(int64_t n, int kp) {
  int64_t g = (n * kp + kNT - 1) / kNT;
  if (g > 1024) g = 1024;
  if (g < 1) g = 1;
  return (unsigned)g;
}

// ---- V-cycle ---------------------------------------------------------------------

struct Smoother {
  int type;        // 0 Jacobi, 1 Chebyshev
  double omega;    // Jacobi weight
  double lmin, lmax;
};

Smoother smoother_for(const Handle& h, const Level& L) {
  Smoother S;
  S.type = h.prm.smootherType;
  S.omega = h.prm.smootherWeight * (4.0 / 3.0) / L.spec.rho;
  // Chebyshev steps keep the V-cycle definite up to lmax + lmin.  Over 292
  // levels of lognormal problems (65^2 to 161^3, sigma 0.5 to 3) the largest
  // eigenvalue came to 1.020 lmax at most, by 1.1 rho alone to 1.17.
  S.lmax = std::max(1.1 * L.spec.rho, L.spec.top);
  S.lmin = S.lmax / 30.0;
  return S;
}

// Bytes of the stored matrix one SpMV with k columns reads: a value and a
// column index per nonzero; the sliced-ELL copy (one column) stores 2-byte
// column codes in its compact slices.  Padding is not counted.
template <typename T>
double matrix_bytes(const Csr& A, int k) {
  const bool sell = k == 1 && A.nslices > 0;
  const double nd = sell ? (double)A.nnz_sdiag : 0.0;  // diagonal outside the slices: no column code
  if (sell && A.lds.bs > 0)  // 16-bit LDS indices, and each block's column list
    return (double)A.nnz * sizeof(T) + 2.0 * ((double)A.nnz - nd) + 4.0 * (double)A.lds.lcols.size();
  const double nc = sell ? (double)A.nnz_compact : 0.0;
  return (double)A.nnz * sizeof(T) + 2.0 * nc + 4.0 * ((double)A.nnz - nd - nc);
}

template <typename T>
void fill_zero(T* p, int64_t n, hipStream_t s);
template <>
void fill_zero<double>(double* p, int64_t n, hipStream_t s) { dev_fill_f64(p, 0.0, (size_t)n, s); }
template <>
void fill_zero<float>(float* p, int64_t n, hipStream_t s) { dev_fill_f32(p, 0.0f, (size_t)n, s); }

// nu steps of the smoother from x = 0 (zero == true) or from the given x.
// Buffers x and t ping-pong; returns the buffer that holds the result.
// Fused FP64 ends of a mixed-precision level-0 smoother (one column, sliced
// ELL): the first step reads the Krylov residual r64 (and stores fl32(r64) in
// b32 for the later steps), the last step writes z64 and r64.z64 partials.
struct Level0Io {
  const double* r64 = nullptr;
  float* b32 = nullptr;
  double* z64 = nullptr;
  double* partials = nullptr;
  unsigned nb = 0;  // partials written by the last step
};

template <typename T>
bool fused_out(const Level0Io* io, const Csr& A, int k) {
  return std::is_same<T, float>::value && io && io->z64 && k == 1 && A.nslices > 0 && A.s32.size() > 0 &&
         A.srow.size() == 0 && A.sell_g == 1;
}

// The last level-0 smoothing step for k > 1 columns with r.z partials
// (io->r64 and io->partials, no io->z64) on the staged copy
template <typename T>
bool multi_out(const Level0Io* io, const Csr& A, int k) {
  return io && io->r64 && io->partials && !io->z64 && k > 1 && k <= 64 && multi_staged<T>(A, k) && A.srow.size() == 0;
}

// The same for one column of an FP64 V-cycle
template <typename T>
bool rz_out(const Level0Io* io, const Csr& A, int k) {
  return std::is_same<T, double>::value && io && io->partials && k == 1 && A.nslices > 0 && A.s64.size() > 0 &&
         A.lds.bs > 0 && A.srow.size() == 0;
}

// nu steps of the smoother from x = 0 (zero == true) or from the given x.
// Buffers x and t ping-pong; returns the buffer that holds the result (with
// io->z64 set, the last step writes there instead and nullptr is returned;
// with multi_out and rz_out, the last step also writes the r.z partials).
// first_done: the first step from zero is already in x (and d), taken by the
// restriction that produced b.
template <typename T>
T* smooth(Handle& h, int l, const Csr& A, const T* b, T* x, T* t, T* d, int nu, bool zero, int k,
          Level0Io* io = nullptr, bool first_done = false) {
  Level& L = *h.H.levels[l];
  hipStream_t s = h.stream;
  const T* dinv = dinv_of<T>(L);
  Smoother S = smoother_for(h, L);
  const bool prof = h.profiling && l == 0;
  // algorithmic bytes of one sweep: the matrix and the per-row vectors
  // (Jacobi: x, b, dinv, x_new; Chebyshev: + d read and write)
  const double sweep_bytes = matrix_bytes<T>(A, k) + (double)A.n * sizeof(T) * (S.type ? 6.0 : 4.0) * k;
  // fused last step: x, b, dinv (+ d) in FP32, r read and z written in FP64
  const double out_bytes = matrix_bytes<T>(A, k) + (double)A.n * (4.0 * (S.type ? 4.0 : 3.0) + 16.0);
  if (nu <= 0) {
    // a fill kernel, not a memset: this may run inside a captured graph
    if (zero) fill_zero<T>(x, A.n * k, s);
    return x;
  }
  const bool in64 = zero && io && io->r64 && std::is_same<T, float>::value && k == 1;
  const bool out64 = !zero && fused_out<T>(io, A, k);
  const bool outk = !zero && multi_out<T>(io, A, k);
  const bool outrz = !zero && rz_out<T>(io, A, k);
  auto first_step = [&](T* xo, T* dout, double c) {
    if (in64) {
      scale_in_kernel<<<grid_for(A.n, 256), 256, 0, s>>>(A.n, (const float*)dinv, io->r64, io->b32, (float*)xo,
                                                          (float*)dout, (float)c);
    } else {
      scale_dinv_kernel<T, T, T><<<grid_for(A.n * k, 256), 256, 0, s>>>(A.n, k, dinv, b, xo, dout, (T)c);
    }
    HIP_LAUNCH_CHECK();
  };
  auto last_step = [&](int mode, T* cur, double c1, double c2) {
    if (A.lds.bs > 0) {
      const size_t lds = sizeof(float) * (size_t)A.lds.maxc;
      lds_launch(A, 4, [&](auto head, unsigned nb, unsigned nt) {
        if (mode == kJacobi)
          sell_lds_out_kernel<kJacobi, head.value><<<nb, nt, lds, s>>>(
              A.n, A.nslices, sell_view(A), lds_view(A.lds), A.s32.get(), (const float*)cur, (const float*)b,
              (const float*)dinv, (const float*)d, (float)c1, (float)c2, io->r64, io->z64, io->partials);
        else
          sell_lds_out_kernel<kCheb, head.value><<<nb, nt, lds, s>>>(
              A.n, A.nslices, sell_view(A), lds_view(A.lds), A.s32.get(), (const float*)cur, (const float*)b,
              (const float*)dinv, (const float*)d, (float)c1, (float)c2, io->r64, io->z64, io->partials);
        io->nb = nb;
      });
      HIP_LAUNCH_CHECK();
      return;
    }
    const unsigned g = grid_for(A.nslices, kNT / 64);
    if (mode == kJacobi)
      sell_smooth_out_kernel<kJacobi><<<g, kNT, 0, s>>>(A.n, A.nslices, sell_view(A), A.s32.get(), (const float*)cur,
                                                         (const float*)b, (const float*)dinv, (const float*)d,
                                                         (float)c1, (float)c2, io->r64, io->z64, io->partials);
    else
      sell_smooth_out_kernel<kCheb><<<g, kNT, 0, s>>>(A.n, A.nslices, sell_view(A), A.s32.get(), (const float*)cur,
                                                       (const float*)b, (const float*)dinv, (const float*)d, (float)c1,
                                                       (float)c2, io->r64, io->z64, io->partials);
    HIP_LAUNCH_CHECK();
    io->nb = g;
  };
  // the last step into xn with the r.z partials (outk, outrz)
  auto last_rz = [&](auto mode, const T* cur, T* xn, double c1, double c2) {
    if (outk) {
      launch_lds_multi<T, mode.value, 2>(A, k, cur, nullptr, b, dinv, d, xn, (T)c1, (T)c2, io->r64, io->partials, s);
      io->nb = multi_blocks(A);
    } else if constexpr (std::is_same<T, double>::value) {
      lds_launch(A, sizeof(T), [&](auto head, unsigned nb, unsigned nt) {
        sell_lds_rz_kernel<mode.value, head.value><<<nb, nt, sizeof(T) * (size_t)A.lds.maxc, s>>>(
            A.n, A.nslices, sell_view(A), lds_view(A.lds), A.s64.get(), cur, b, dinv, d, xn, c1, c2, io->partials);
        io->nb = nb;
      });
    }
    HIP_LAUNCH_CHECK();
  };
  T* cur = x;
  T* nxt = t;
  int step = 0;
  if (S.type == 0) {
    const T w = (T)S.omega;
    if (zero) {
      if (!first_done) first_step(cur, nullptr, S.omega);
      step = 1;
    }
    for (; step < nu; ++step) {
      if (out64 && step == nu - 1) {
        ProfScope ps(h, prof ? "smooth_l0_out" : "", out_bytes);
        last_step(kJacobi, cur, S.omega, 0.0);
        return nullptr;
      }
      ProfScope ps(h, prof ? "smooth_l0" : "", sweep_bytes);
      if ((outk || outrz) && step == nu - 1) {
        last_rz(std::integral_constant<int, kJacobi>{}, cur, nxt, S.omega, 0.0);
        return nxt;
      }
      spmv_op<T, kJacobi>(A, k, cur, nullptr, b, dinv, nullptr, nxt, w, T(0), s);
      T* tmp = cur; cur = nxt; nxt = tmp;
    }
    return cur;
  }
  // Chebyshev on D^-1 A over [lmin, lmax]
  const double theta = 0.5 * (S.lmax + S.lmin), delta = 0.5 * (S.lmax - S.lmin);
  const double sigma = theta / delta;
  double rho_old = 1.0 / sigma;
  if (zero) {
    if (!first_done) first_step(cur, d, 1.0 / theta);
    step = 1;
  }
  for (; step < nu; ++step) {
    double c1, c2;
    if (step == 0) {
      c1 = 0.0;
      c2 = 1.0 / theta;
    } else {
      double rho_new = 1.0 / (2.0 * sigma - rho_old);
      c1 = rho_new * rho_old;
      c2 = 2.0 * rho_new / delta;
      rho_old = rho_new;
    }
    if (out64 && step == nu - 1) {
      ProfScope ps(h, prof ? "smooth_l0_out" : "", out_bytes);
      last_step(kCheb, cur, c1, c2);
      return nullptr;
    }
    ProfScope ps(h, prof ? "smooth_l0" : "", sweep_bytes);
    if ((outk || outrz) && step == nu - 1) {
      last_rz(std::integral_constant<int, kCheb>{}, cur, nxt, c1, c2);
      return nxt;
    }
    spmv_op<T, kCheb>(A, k, cur, nullptr, b, dinv, d, nxt, (T)c1, (T)c2, s);
    T* tmp = cur; cur = nxt; nxt = tmp;
  }
  return cur;
}

// b_{l+1} = R r.  When level l+1 is smoothed from zero (not the coarsest
// level) the same pass takes its first smoothing step, x = c D^-1 b (and
// d = x for Chebyshev), as smooth() would; returns whether it did.
template <typename T>
bool restrict_first(Handle& h, int l, const Csr& R, const T* r, int k) {
  Hierarchy& H = h.H;
  Level& N = *H.levels[l + 1];
  T* bc = LV<T>::b(N);
  if (l + 1 == H.coarse || h.prm.preInnerIters < 1) {
    spmv_op<T, kAssign>(R, k, r, bc, nullptr, (const T*)nullptr, nullptr, nullptr, T(0), T(0), h.stream);
    return false;
  }
  const Smoother S = smoother_for(h, N);
  const double c = S.type ? 1.0 / (0.5 * (S.lmax + S.lmin)) : S.omega;
  spmv_op<T, kAssignScale>(R, k, r, bc, nullptr, dinv_of<T>(N), S.type ? LV<T>::d(N) : nullptr, LV<T>::x(N), (T)c,
                           T(0), h.stream);
  return true;
}

// Chebyshev coefficients of step `step` of a smoother on [lmin, lmax]
struct ChebSeq {
  double theta, delta, sigma, rho_old;
  explicit ChebSeq(const Smoother& S)
      : theta(0.5 * (S.lmax + S.lmin)), delta(0.5 * (S.lmax - S.lmin)), sigma(theta / delta), rho_old(delta / theta) {}
  void next(int step, double& c1, double& c2) {
    if (step == 0) {
      c1 = 0.0;
      c2 = 1.0 / theta;
    } else {
      const double rho_new = 1.0 / (2.0 * sigma - rho_old);
      c1 = rho_new * rho_old;
      c2 = 2.0 * rho_new / delta;
      rho_old = rho_new;
    }
  }
};

// ---- the V-cycle's small levels in one launch --------------------------------------
// One block restricts the residual of the level above, runs the V-cycle of
// the levels below it and solves the coarsest level, with the levels'
// matrices and vectors in LDS.  Level by level these are some ten launches,
// each a few microseconds of launch and load latency for a few thousand
// entries: 65^2 (297 and 21 rows, FP64) 33 us in ten launches, 20 us here;
// 1003 x 701 (300 and 19 rows below five levels, FP32) 50 -> 27 us; 97^3
// (restriction and the 59-row solve only) 16 -> 9.5 us.  A phase is a chain of
// LDS reads per row, about 1.5 us: with the matrices left in L2 it took 2 us,
// and with 512 or 256 threads the launch takes 24 and 33 us at 65^2.
constexpr int kTailLevels = 6;
constexpr int kTailSteps = 8;
constexpr int kTailNT = 1024;
constexpr size_t kTailLds = 150 * 1024;
// What stays in memory is streamed by one CU, so it has to be little: entries
// of the restriction into the first level, rows of the coarsest level (its
// inverse; 13^3, 100 rows: the launch takes 12 us against 5 for the two that
// use the whole chip)
constexpr int64_t kTailRnnz = 16384;
constexpr int64_t kTailCoarse = 64;
// rows of a smoothed level: 260 x 240 FP64 solves in 4.39 ms with its
// level of 250 to 480 rows in here, 4.90 with it in launches; larger ones mostly fall to
// the restriction's limit above (a limit of 1024 rows times the same from 300 x
// 280 to 500 x 480, 13^3 to 49^3)
constexpr int64_t kTailRows = 480;

template <typename T>
struct TailCsr {
  const int32_t* rp;
  const int32_t* ci;
  const T* v;
  int n, nnz, lg;       // rows, entries, log2 of the lanes per row
  int o_v, o_rp, o_ci;  // byte offsets of its copy in LDS
};

template <typename T>
struct TailLevel {
  TailCsr<T> A, P, R;
  const T* dinv;
  int o_dinv, o_vec;  // LDS: D^-1; x, t, b, d, r
  T c0;               // first step from zero
  T pre1[kTailSteps], pre2[kTailSteps], post1[kTailSteps], post2[kTailSteps];
};

template <typename T>
struct TailArgs {
  int nlev;  // smoothed levels, then the coarsest
  int type, npre, npost;
  TailCsr<T> R;        // restriction into the first level (in memory)
  const T* r;          // residual above it
  T* x;                // its result
  const double* cinv;  // the coarsest level's inverse
  int nc, o_coarse;    // LDS: its x and b
  TailLevel<T> lev[kTailLevels];
};

// f(row, (M x)_row) for every row, xs(j) = x_j; the block's threads in groups
// of 2^lg lanes per row
template <typename T, typename RP, typename CI, typename X, typename F>
__device__ __forceinline__ void tail_rows(int n, int lg, const RP* rp, const CI* ci, const T* v, X xs, F f) {
  const int g = 1 << lg, lane = threadIdx.x & (g - 1);
  for (int row = threadIdx.x >> lg; row < n; row += kTailNT >> lg) {
    const int e = rp[row + 1];
    int q = rp[row] + lane;
    T acc = T(0);
    for (; q + 3 * g < e; q += 4 * g) {
      const int j0 = ci[q], j1 = ci[q + g], j2 = ci[q + 2 * g], j3 = ci[q + 3 * g];
      const T v0 = v[q], v1 = v[q + g], v2 = v[q + 2 * g], v3 = v[q + 3 * g];
      const T x0 = xs(j0), x1 = xs(j1), x2 = xs(j2), x3 = xs(j3);
      acc += v0 * x0;
      acc += v1 * x1;
      acc += v2 * x2;
      acc += v3 * x3;
    }
    for (; q < e; q += g) acc += v[q] * xs(ci[q]);
    for (int off = g >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) f(row, acc);
  }
  __syncthreads();
}

template <typename T>
__global__ void __launch_bounds__(kTailNT) tail_kernel(TailArgs<T> S) {
  extern __shared__ unsigned char lds[];
  auto put = [&](const TailCsr<T>& M) {
    T* v = reinterpret_cast<T*>(lds + M.o_v);
    int* rp = reinterpret_cast<int*>(lds + M.o_rp);
    uint16_t* ci = reinterpret_cast<uint16_t*>(lds + M.o_ci);
    for (int t = threadIdx.x; t < M.nnz; t += kTailNT) {
      v[t] = M.v[t];
      ci[t] = (uint16_t)M.ci[t];
    }
    for (int t = threadIdx.x; t <= M.n; t += kTailNT) rp[t] = M.rp[t];
  };
  for (int l = 0; l < S.nlev; ++l) {
    const TailLevel<T>& L = S.lev[l];
    put(L.A);
    put(L.P);
    put(L.R);
    T* dinv = reinterpret_cast<T*>(lds + L.o_dinv);
    for (int t = threadIdx.x; t < L.A.n; t += kTailNT) dinv[t] = L.dinv[t];
  }
  // f over the rows of a staged matrix times the LDS vector x
  auto rows = [&](const TailCsr<T>& M, const T* x, auto f) {
    tail_rows(M.n, M.lg, reinterpret_cast<const int*>(lds + M.o_rp), reinterpret_cast<const uint16_t*>(lds + M.o_ci),
              reinterpret_cast<const T*>(lds + M.o_v), [=](int j) { return x[j]; }, f);
  };
  // level l's x, t, b, d, r; the coarsest level's x and b
  enum { VX = 0, VT = 1, VB = 2, VD = 3, VR = 4 };
  auto vec = [&](int l, int which) { return reinterpret_cast<T*>(lds + S.lev[l].o_vec) + which * S.lev[l].A.n; };
  T* const cx = reinterpret_cast<T*>(lds + S.o_coarse);
  T* const cb = cx + S.nc;
  {
    T* b = S.nlev > 0 ? vec(0, VB) : cb;
    const T* r = S.r;
    tail_rows(S.R.n, S.R.lg, S.R.rp, S.R.ci, S.R.v, [=](int j) { return r[j]; }, [=](int row, T a) { b[row] = a; });
  }
  // one smoother step: xo = x + its correction, d updated
  auto smooth = [&](const TailLevel<T>& L, const T* x, T* xo, const T* b, T* d, T c1, T c2) {
    const T* dinv = reinterpret_cast<const T*>(lds + L.o_dinv);
    const int type = S.type;
    rows(L.A, x, [=](int row, T a) {
      if (type == 0) {
        xo[row] = x[row] + c1 * dinv[row] * (b[row] - a);
      } else {
        const T r = dinv[row] * (b[row] - a);
        const T dn = (c1 != T(0) ? c1 * d[row] : T(0)) + c2 * r;
        d[row] = dn;
        xo[row] = x[row] + dn;
      }
    });
  };
  const int moves = S.npre > 1 ? S.npre - 1 : 0;  // steps that move x to t or back before the correction
  for (int l = 0; l < S.nlev; ++l) {
    const TailLevel<T>& L = S.lev[l];
    T *x = vec(l, VX), *t = vec(l, VT), *b = vec(l, VB), *d = vec(l, VD), *r = vec(l, VR);
    const T* dinv = reinterpret_cast<const T*>(lds + L.o_dinv);
    for (int i = threadIdx.x; i < L.A.n; i += kTailNT) {
      const T v = S.npre > 0 ? L.c0 * dinv[i] * b[i] : T(0);
      x[i] = v;
      d[i] = v;
    }
    __syncthreads();
    for (int st = 1; st <= moves; ++st) {
      smooth(L, x, t, b, d, L.pre1[st], L.pre2[st]);
      T* w = x; x = t; t = w;
    }
    rows(L.A, x, [=](int row, T a) { r[row] = b[row] - a; });
    T* bn = l + 1 < S.nlev ? vec(l + 1, VB) : cb;
    rows(L.R, r, [=](int row, T a) { bn[row] = a; });
  }
  // coarsest level: FP64 sums in every precision, a wavefront per row
  {
    constexpr int kRows = (int)kTailCoarse / (kTailNT / 64);  // rows of a wavefront, loaded together
    const int j = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double acc[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const int row = wave + i * (kTailNT / 64);
      acc[i] = row < S.nc && j < S.nc ? S.cinv[(int64_t)row * S.nc + j] * (double)cb[j] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const int row = wave + i * (kTailNT / 64);
      const double sum = wave_sum(acc[i]);
      if (row < S.nc && j == 0) {
        cx[row] = (T)sum;
        if (S.nlev == 0) S.x[row] = (T)sum;
      }
    }
    __syncthreads();
  }
  for (int l = S.nlev - 1; l >= 0; --l) {
    const TailLevel<T>& L = S.lev[l];
    T *x = vec(l, (moves & 1) ? VT : VX), *t = vec(l, (moves & 1) ? VX : VT), *b = vec(l, VB), *d = vec(l, VD);
    const T* xc = l + 1 < S.nlev ? vec(l + 1, ((moves + S.npost) & 1) ? VT : VX) : cx;
    rows(L.P, xc, [=](int row, T a) { x[row] += a; });
    for (int st = 0; st < S.npost; ++st) {
      smooth(L, x, t, b, d, L.post1[st], L.post2[st]);
      T* w = x; x = t; t = w;
    }
    if (l == 0)
      for (int i = threadIdx.x; i < L.A.n; i += kTailNT) S.x[i] = x[i];
  }
}

// lanes per row: the block's threads over the rows, at least one entry a lane
template <typename T>
TailCsr<T> tail_csr(const Csr& M) {
  const double avg = M.n ? (double)M.nnz / (double)M.n : 1.0;
  int lg = 0;
  while (lg < 6 && (M.n << (lg + 1)) <= kTailNT && avg > (double)(1 << lg)) ++lg;
  return TailCsr<T>{M.rp.get(), M.ci.get(), vals_of<T>(M), (int)M.n, (int)M.nnz, lg, 0, 0, 0};
}

// Arguments of the tail from level l (R: the restriction into it); returns its
// LDS bytes, 0 when the levels do not fit.
template <typename T>
size_t plan_tail(const Handle& h, int l, const Csr& R, TailArgs<T>& S) {
  const Hierarchy& H = h.H;
  S.nlev = H.coarse - l;
  S.type = h.prm.smootherType;
  S.npre = h.prm.preInnerIters;
  S.npost = h.prm.postInnerIters * (h.prm.postRelaxes > 0 ? h.prm.postRelaxes : 1);
  if (l < 1 || S.nlev < 0 || S.nlev > kTailLevels || S.npre > kTailSteps || S.npost > kTailSteps) return 0;
  if (R.nnz > kTailRnnz || H.nc > kTailCoarse) return 0;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t o = at;
    at = (at + bytes + 15) & ~(size_t)15;
    return (int)o;
  };
  S.nc = (int)H.nc;
  S.o_coarse = take(2 * sizeof(T) * (size_t)H.nc);
  auto place = [&](const Csr& M) {
    TailCsr<T> c = tail_csr<T>(M);
    c.o_v = take(sizeof(T) * (size_t)M.nnz);
    c.o_rp = take(sizeof(int) * (size_t)(M.n + 1));
    c.o_ci = take(sizeof(uint16_t) * (size_t)M.nnz);
    return c;
  };
  for (int j = l; j < H.coarse; ++j) {
    const Level& L = *H.levels[j];
    if (L.A.n > kTailRows || L.A.nnz * (int64_t)sizeof(T) > (int64_t)kTailLds) return 0;
    TailLevel<T>& t = S.lev[j - l];
    t.A = place(L.A);
    t.P = place(L.P);
    t.R = place(L.R);
    t.dinv = dinv_of<T>(L);
    t.o_dinv = take(sizeof(T) * (size_t)L.A.n);
    t.o_vec = take(5 * sizeof(T) * (size_t)L.A.n);
    if (at > kTailLds) return 0;
    const Smoother sm = smoother_for(h, L);
    ChebSeq a(sm), b(sm);
    t.c0 = (T)(sm.type ? 1.0 / a.theta : sm.omega);
    for (int st = 0; st < kTailSteps; ++st) {
      double c1 = sm.omega, c2 = 0.0;
      if (sm.type) a.next(st, c1, c2);
      t.pre1[st] = (T)c1;
      t.pre2[st] = (T)c2;
      c1 = sm.omega;
      c2 = 0.0;
      if (sm.type) b.next(st, c1, c2);
      t.post1[st] = (T)c1;
      t.post2[st] = (T)c2;
    }
  }
  S.R = tail_csr<T>(R);
  S.cinv = H.cinv64.get();
  return at;
}

// Cycle types (cycleType): 0 V; 1 W, whose coarse correction is two W-cycles
// of the next level, the second from the first's result (cycles/wcycle.h);
// 2 F, whose coarse correction is an F-cycle of the next level followed by a
// V-cycle from its result (the textbook F-cycle; cycles/fcycle.h writes a
// W-cycle first).  3 (K) is a V-cycle: the reference dispatches K_CYCLE as
// the outer CG_Flex_Cycle itself (cycles/cycle.h:34-36, amg.cu:160-165).
constexpr int kCycleV = 0, kCycleW = 1, kCycleF = 2;

int cycle_type(const Handle& h) {
  const int c = h.prm.cycleType;
  return (c == kCycleW || c == kCycleF) ? c : kCycleV;
}

template <typename T>
T* vcycle(Handle& h, int l, const T* b, int k, Level0Io* io = nullptr, bool first_done = false, int type = kCycleV,
          T* x0 = nullptr);

// Coarse correction of level l, the right-hand side already restricted into
// level l+1's b: one cycle of level l+1 (V), or two (W: W then W; F: F then
// V).  Returns level l+1's buffer holding the correction.
template <typename T>
T* coarse_correction(Handle& h, int l, int k, bool next_first, int type) {
  Level& N = *h.H.levels[l + 1];
  T* xc = vcycle<T>(h, l + 1, LV<T>::b(N), k, nullptr, next_first, type);
  if (type != kCycleV && l + 1 != h.H.coarse)
    xc = vcycle<T>(h, l + 1, LV<T>::b(N), k, nullptr, false, type == kCycleW ? kCycleW : kCycleV, xc);
  return xc;
}

// Level l's coarse correction from its residual r: restriction by R and the
// cycle of level l+1, in one launch where the levels below are small
template <typename T>
T* correction(Handle& h, int l, const Csr& R, const T* r, int k, int type) {
  if (k == 1 && type == kCycleV) {
    TailArgs<T> S{};
    if (const size_t bytes = plan_tail<T>(h, l + 1, R, S)) {
      S.r = r;
      S.x = LV<T>::x(*h.H.levels[l + 1]);
      tail_kernel<T><<<1, kTailNT, bytes, h.stream>>>(S);
      HIP_LAUNCH_CHECK();
      return S.x;
    }
  }
  const bool next_first = restrict_first<T>(h, l, R, r, k);
  return coarse_correction<T>(h, l, k, next_first, type);
}

// One cycle of the given type on level l for the right-hand side b (level l
// vectors, k columns), from zero or (x0, one of level l's x / t buffers) from
// x0; returns the buffer holding the result (nullptr when io->z64 received
// it).  first_done: restrict_first took the first pre-smoothing step.
template <typename T>
T* vcycle(Handle& h, int l, const T* b, int k, Level0Io* io, bool first_done, int type, T* x0) {
  Hierarchy& H = h.H;
  Level& L = *H.levels[l];
  hipStream_t s = h.stream;
  const Csr& A = level_A(h, l);
  if (l == H.coarse) {  // the direct solve does not depend on a start
    coarse_kernel<T><<<(unsigned)H.nc, 64, 0, s>>>(H.nc, k, H.cinv64.get(), b, LV<T>::x(L));
    HIP_LAUNCH_CHECK();
    return LV<T>::x(L);
  }
  if (x0 && (io || first_done)) fail(FEM_ERR_STATE, "a cycle from a given start takes no fused ends");
  T* x = x0 ? x0 : LV<T>::x(L);
  T* t = (x == LV<T>::x(L)) ? LV<T>::t(L) : LV<T>::x(L);
  T* r = LV<T>::r(L);
  T* d = LV<T>::d(L);
  const int nu_pre = h.prm.preInnerIters;
  const int nu_post = h.prm.postInnerIters * (h.prm.postRelaxes > 0 ? h.prm.postRelaxes : 1);
  T* cur = smooth<T>(h, l, A, b, x, t, d, nu_pre, x0 == nullptr, k, x0 ? nullptr : io, first_done);
  T* oth = (cur == x) ? t : x;
  {
    ProfScope ps(h, (h.profiling && l == 0) ? "resid_l0" : "", matrix_bytes<T>(A, k) + 3.0 * A.n * k * sizeof(T));
    spmv_op<T, kResid>(A, k, cur, r, b, (const T*)nullptr, nullptr, nullptr, T(0), T(0), s);
  }
  T* xc = correction<T>(h, l, L.R, r, k, type);
  spmv_op<T, kAdd>(L.P, k, xc, cur, nullptr, (const T*)nullptr, nullptr, nullptr, T(0), T(0), s);
  cur = smooth<T>(h, l, A, b, cur, oth, d, nu_post, false, k, io);
  return cur;
}

// Precision 2, one column: the level-0 part of the V-cycle in y = D^1/2 x (the
// same V-cycle as the FP32 one: Chebyshev/Jacobi on a matrix similar to
// D^-1 A, restriction by (D^1/2 P)^T, prolongation by D^1/2 P), with the
// FP64 residual in and z = D^-1/2 y out.  Returns the count of r.z partials.
unsigned vcycle0_half(Handle& h, const double* r64, double* z64, double* partials) {
  Hierarchy& H = h.H;
  Level& L0 = *H.levels[0];
  hipStream_t s = h.stream;
  const Csr& O = H.ah;
  const int64_t n = O.n;
  float* bh = L0.b32.get();
  float* rr = L0.r32.get();
  float* d = L0.d32.get();
  float* cur = L0.x32.get();
  float* nxt = L0.t32.get();
  const Smoother S = smoother_for(h, L0);
  const int nu_pre = h.prm.preInnerIters;
  const int nu_post = h.prm.postInnerIters * (h.prm.postRelaxes > 0 ? h.prm.postRelaxes : 1);
  const unsigned g = grid_for(O.nslices, kNT / 64);
  const SellView V = sell_view(O);
  // LDS-staged copy when its lists exist: one block per O.lds.bs slices
  const bool staged = O.lds.bs > 0;
  const LdsView LV_ = staged ? lds_view(O.lds) : LdsView{};
  const unsigned gl = staged ? (unsigned)((O.nslices + O.lds.bs - 1) / O.lds.bs) : 0;
  const size_t ldsb = staged ? sizeof(float) * (size_t)O.lds.maxc : 0;
  // algorithmic bytes: FP16 value + column code per off-diagonal, and y, b^, diag (+ d r/w), y_new
  const double mbytes = staged ? 2.0 * (double)O.nnz + 2.0 * (double)O.nnz + 4.0 * (double)O.lds.lcols.size()
                               : 2.0 * (double)O.nnz + 2.0 * (double)O.nnz_compact +
                                     4.0 * ((double)O.nnz - O.nnz_compact);
  const double step_bytes = mbytes + 4.0 * n * (S.type ? 6.0 : 4.0);
  const bool prof = h.profiling;
  auto staged_step = [&](auto mode, float c1, float c2) {
    lds_launch(O, 2, [&](auto head, unsigned nb, unsigned nt) {
      sell_half_lds_kernel<mode.value, head.value><<<nb, nt, ldsb, s>>>(n, O.nslices, V, LV_, O.sh.get(),
                                                                       H.ah_diag.get(), cur, bh, rr, d, nxt, c1, c2);
    });
  };
  auto staged_out = [&](auto mode, float c1, float c2) {
    lds_launch(O, 2, [&](auto head, unsigned nb, unsigned nt) {
      sell_half_lds_out_kernel<mode.value, head.value><<<nb, nt, ldsb, s>>>(
          n, O.nslices, V, LV_, O.sh.get(), H.ah_diag.get(), H.ah_s.get(), cur, bh, d, c1, c2, r64, z64, partials);
    });
  };
  using ModeResid = std::integral_constant<int, kResid>;
  using ModeJacobi = std::integral_constant<int, kJacobi>;
  using ModeCheb = std::integral_constant<int, kCheb>;
  auto step = [&](int mode, double c1, double c2) {
    ProfScope ps(h, prof ? "smooth_l0_h" : "", step_bytes);
    if (staged && mode == kJacobi)
      staged_step(ModeJacobi{}, (float)c1, 0.0f);
    else if (staged)
      staged_step(ModeCheb{}, (float)c1, (float)c2);
    else if (mode == kJacobi)
      sell_half_kernel<kJacobi><<<g, kNT, 0, s>>>(n, O.nslices, V, O.sh.get(), H.ah_diag.get(), cur, bh, nullptr,
                                                  nullptr, nxt, (float)c1, 0.0f);
    else
      sell_half_kernel<kCheb><<<g, kNT, 0, s>>>(n, O.nslices, V, O.sh.get(), H.ah_diag.get(), cur, bh, nullptr, d,
                                                nxt, (float)c1, (float)c2);
    HIP_LAUNCH_CHECK();
    std::swap(cur, nxt);
  };
  // pre-smoothing from y = 0
  ChebSeq cs(S);
  scale_in_half_kernel<<<grid_for(n, 256), 256, 0, s>>>(n, H.ah_s.get(), r64, bh, cur, S.type ? d : nullptr,
                                                         (float)(S.type ? 1.0 / cs.theta : S.omega));
  HIP_LAUNCH_CHECK();
  for (int st = 1; st < nu_pre; ++st) {
    double c1 = S.omega, c2 = 0.0;
    if (S.type) cs.next(st, c1, c2);
    step(S.type ? kCheb : kJacobi, c1, c2);
  }
  // residual, restriction, coarse correction, prolongation
  if (staged)
    staged_step(ModeResid{}, 0.0f, 0.0f);
  else
    sell_half_kernel<kResid><<<g, kNT, 0, s>>>(n, O.nslices, V, O.sh.get(), H.ah_diag.get(), cur, bh, rr, nullptr,
                                                nullptr, 0.0f, 0.0f);
  HIP_LAUNCH_CHECK();
  float* xc = correction<float>(h, 0, H.rh, rr, 1, cycle_type(h));
  spmv_op<float, kAdd>(H.ph, 1, xc, cur, nullptr, (const float*)nullptr, nullptr, nullptr, 0.0f, 0.0f, s);
  // post-smoothing; the last step writes z and the r.z partials
  ChebSeq cp(S);
  for (int st = 0; st < nu_post; ++st) {
    double c1 = S.omega, c2 = 0.0;
    if (S.type) cp.next(st, c1, c2);
    if (st < nu_post - 1) {
      step(S.type ? kCheb : kJacobi, c1, c2);
      continue;
    }
    ProfScope ps(h, prof ? "smooth_l0_h_out" : "", step_bytes + 12.0 * n);
    if (staged) {
      if (S.type)
        staged_out(ModeCheb{}, (float)c1, (float)c2);
      else
        staged_out(ModeJacobi{}, (float)c1, 0.0f);
      HIP_LAUNCH_CHECK();
      continue;
    }
    if (S.type)
      sell_half_out_kernel<kCheb><<<g, kNT, 0, s>>>(n, O.nslices, V, O.sh.get(), H.ah_diag.get(), H.ah_s.get(), cur,
                                                    bh, d, (float)c1, (float)c2, r64, z64, partials);
    else
      sell_half_out_kernel<kJacobi><<<g, kNT, 0, s>>>(n, O.nslices, V, O.sh.get(), H.ah_diag.get(), H.ah_s.get(),
                                                      cur, bh, nullptr, (float)c1, 0.0f, r64, z64, partials);
    HIP_LAUNCH_CHECK();
  }
  return staged ? gl : g;
}

// Where one application of the preconditioner left z = M r.
struct PrecOut {
  const double* z64 = nullptr;  // FP64 z: the caller's buffer or a level-0 work vector
  const float* z32 = nullptr;   // or the FP32 V-cycle result (exact in FP64)
  unsigned nb = 0;              // r.z partials written by the fused level-0 ends
};

// One column, mixed precision, level 0 smoothed before and after the coarse
// correction, sliced ELL: the FP64 <-> FP32 conversions are fused into the
// first and last level-0 smoothing steps, and the last one also writes
// per-block partials of r.z.
bool fused_level0(const Handle& h, int k, bool partials) {
  const int nu_post = h.prm.postInnerIters * (h.prm.postRelaxes > 0 ? h.prm.postRelaxes : 1);
  return partials && h.H.precision >= 1 && k == 1 && h.H.coarse > 0 && h.prm.preInnerIters >= 1 && nu_post >= 1 &&
         h.A.nslices > 0 && h.A.s32.size() > 0 && h.A.sell_g == 1;
}

// Outputs of the PCG update for a level-0 V-cycle in T: b = fl32(r) (FP32; an
// FP64 V-cycle reads r), and the smoother's first step from zero, x0 = c0 dinv
// b (and d0 = x0 for Chebyshev).  Off for the FP16 level-0 smoother (its own
// first step) and for hierarchies without level-0 smoothing.
template <typename T>
struct First0 {
  bool on = false;
  T* b = nullptr;
  const T* dinv = nullptr;
  T* x0 = nullptr;
  T* d0 = nullptr;
  T c0 = T(0);
};

template <typename T>
First0<T> first0_for(Handle& h, int k) {
  constexpr bool f32 = std::is_same<T, float>::value;
  First0<T> f;
  if ((h.H.precision >= 1) != f32 || h.H.coarse <= 0 || h.prm.preInnerIters < 1) return f;
  if (h.H.precision == 2 && fused_level0(h, k, true) && h.H.ah.nslices > 0) return f;
  Level& L0 = *h.H.levels[0];
  const Smoother S = smoother_for(h, L0);
  if (f32) f.b = LV<T>::b(L0);
  f.dinv = dinv_of<T>(L0);
  f.x0 = LV<T>::x(L0);
  if (S.type == 0) {
    f.c0 = (T)S.omega;
  } else {
    f.c0 = (T)(1.0 / (0.5 * (S.lmax + S.lmin)));
    f.d0 = LV<T>::d(L0);
  }
  f.on = f.dinv != nullptr && f.x0 != nullptr;
  return f.on ? f : First0<T>();
}

// z = M r at level 0 (FP64 r); k columns.  z is written only on the fused
// path; otherwise it is left where the V-cycle put it (no copy).  r32_ready:
// the level-0 FP32 right-hand side already holds fl32(r); first_ready: the
// level-0 smoother's first step from zero is in its x (and d) too.
PrecOut precondition_pcg(Handle& h, const double* r, double* z, int k, double* partials, bool r32_ready,
                         bool first_ready) {
  hipStream_t s = h.stream;
  Level& L0 = *h.H.levels[0];
  const int64_t m = h.A.n * k;
  PrecOut o;
  const int type = cycle_type(h);
  if (h.H.precision == 0) {
    // the last level-0 smoothing step also writes the r.z partials when it
    // runs on the staged copy (o.nb stays 0 otherwise)
    Level0Io io;
    io.r64 = r;
    io.partials = partials;
    o.z64 = vcycle<double>(h, 0, r, k, partials ? &io : nullptr, first_ready, type);
    o.nb = io.nb;
    return o;
  }
  if (fused_level0(h, k, partials != nullptr)) {
    if (h.H.precision == 2 && h.H.ah.nslices > 0) {
      o.nb = vcycle0_half(h, r, z, partials);
    } else {
      Level0Io io;
      io.r64 = r;
      io.b32 = L0.b32.get();
      io.z64 = z;
      io.partials = partials;
      float* res = vcycle<float>(h, 0, L0.b32.get(), 1, &io, first_ready, type);
      if (res || io.nb == 0) fail(FEM_ERR_STATE, "fused level-0 smoother did not write its output");
      o.nb = io.nb;
    }
    o.z64 = z;
    return o;
  }
  if (!r32_ready) {
    convert_kernel<double, float><<<grid_for(m, 256), 256, 0, s>>>(m, r, L0.b32.get());
    HIP_LAUNCH_CHECK();
  }
  // k > 1: the last level-0 smoothing step also writes the r.z partials
  // (when it runs on the sliced copy; o.nb stays 0 otherwise)
  Level0Io io;
  io.r64 = r;
  io.partials = partials;
  o.z32 = vcycle<float>(h, 0, L0.b32.get(), k, (partials && k > 1) ? &io : nullptr, r32_ready && first_ready,
                        type);
  o.nb = io.nb;
  return o;
}

// z = M r into z (FP64); returns the count of r.z partials written (fused path)
unsigned precondition(Handle& h, const double* r, double* z, int k, double* partials = nullptr) {
  hipStream_t s = h.stream;
  const int64_t m = h.A.n * k;
  const PrecOut o = precondition_pcg(h, r, z, k, partials, false, false);
  if (o.z32) {
    convert_kernel<float, double><<<grid_for(m, 256), 256, 0, s>>>(m, o.z32, z);
    HIP_LAUNCH_CHECK();
  } else if (o.z64 != z) {
    copy_kernel<<<grid_for(m, 256), 256, 0, s>>>(m, o.z64, z);
    HIP_LAUNCH_CHECK();
  }
  return o.nb;
}

}  // namespace

namespace {
hipEvent_t take_event(Handle& h) {
  if (!h.ev_pool.empty()) {
    hipEvent_t e = h.ev_pool.back();
    h.ev_pool.pop_back();
    return e;
  }
  hipEvent_t e;
  HIP_CHECK(hipEventCreate(&e));
  return e;
}
}  // namespace

ProfScope::ProfScope(Handle& hh, const char* f, double b) : h(hh), fam(f), bytes(b), on(hh.profiling && f && f[0]) {
  if (!on) return;
  a = take_event(h);
  HIP_CHECK(hipEventRecord(a, h.stream));
}

ProfScope::~ProfScope() {
  if (!on) return;
  hipEvent_t b = take_event(h);
  if (hipEventRecord(b, h.stream) != hipSuccess) return;
  h.pending.push_back(PendingTiming{fam, a, b, bytes});
  if (h.pending.size() >= 8192) flush_profile(h);
}

void flush_profile(Handle& h) {
  if (h.pending.empty()) return;
  HIP_CHECK(hipStreamSynchronize(h.stream));
  for (auto& p : h.pending) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, p.a, p.b) == hipSuccess) {
      KernelStat& st = h.stats[p.fam];
      st.launches += 1;
      st.total_ms += ms;
      st.bytes = p.bytes;
    }
    h.ev_pool.push_back(p.a);
    h.ev_pool.push_back(p.b);
  }
  h.pending.clear();
}

void release_profile_events(Handle& h) {
  for (auto& p : h.pending) {
    (void)hipEventDestroy(p.a);
    (void)hipEventDestroy(p.b);
  }
  h.pending.clear();
  for (auto e : h.ev_pool) (void)hipEventDestroy(e);
  h.ev_pool.clear();
}

void spmv64(const Csr& A, const double* x, double* y, hipStream_t s) {
  spmv_op<double, kAssign>(A, 1, x, y, nullptr, (const double*)nullptr, nullptr, nullptr, 0.0, 0.0, s);
}

void apply_operator_int(Handle& h, const double* x, double* y, int k) {
  spmv_op<double, kAssign>(h.A, k, x, y, nullptr, (const double*)nullptr, nullptr, nullptr, 0.0, 0.0, h.stream);
}

const Csr& level_matrix_of(const Handle& h, int lvl, int which) {
  const Hierarchy& H = h.H;
  if (lvl < 0 || lvl >= (int)H.levels.size()) fail(FEM_ERR_ARG, "level out of range");
  if (which == 0 || which == 3) return level_A(h, lvl);
  if (which != 1 && which != 2) fail(FEM_ERR_ARG, "which: 0 operator, 1 prolongator, 2 restriction");
  if (lvl == H.coarse) fail(FEM_ERR_ARG, "the coarsest level has no prolongator or restriction");
  return which == 1 ? H.levels[lvl]->P : H.levels[lvl]->R;
}

void level_smoother_info(const Handle& h, int lvl, double* rho, double* lmin, double* lmax, double* omega) {
  const Hierarchy& H = h.H;
  if (lvl < 0 || lvl >= (int)H.levels.size()) fail(FEM_ERR_ARG, "level out of range");
  if (lvl == H.coarse) fail(FEM_ERR_ARG, "the coarsest level is solved directly, it has no smoother");
  const Level& L = *H.levels[lvl];
  const Smoother S = smoother_for(h, L);
  if (rho) *rho = L.spec.rho;
  if (lmin) *lmin = S.lmin;
  if (lmax) *lmax = S.lmax;
  if (omega) *omega = S.omega;
}

namespace {
template <typename T>
void smoother_step_t(Handle& h, const Csr& A, const T* dinv, int mode, double c1, double c2, const T* x, const T* b,
                     T* d, T* y) {
  if (mode == 0)
    spmv_op<T, kJacobi>(A, 1, x, nullptr, b, dinv, nullptr, y, (T)c1, T(0), h.stream);
  else
    spmv_op<T, kCheb>(A, 1, x, nullptr, b, dinv, d, y, (T)c1, (T)c2, h.stream);
}
}  // namespace

void smoother_step_int(Handle& h, int lvl, int mode, double c1, double c2, const double* x, const double* b,
                       double* d, double* y) {
  const Hierarchy& H = h.H;
  if (lvl < 0 || lvl >= (int)H.levels.size() || lvl == H.coarse) fail(FEM_ERR_ARG, "level has no smoother");
  if (mode != 0 && mode != 1) fail(FEM_ERR_ARG, "mode: 0 Jacobi, 1 Chebyshev");
  const Csr& A = level_A(h, lvl);
  const Level& L = *H.levels[lvl];
  hipStream_t s = h.stream;
  const int64_t n = A.n;
  if (H.precision == 0) {
    smoother_step_t<double>(h, A, L.dinv64.get(), mode, c1, c2, x, b, d, y);
  } else {
    if (!A.v32.size() || (A.nslices > 0 && !A.s32.size()) || !L.dinv32.size())
      fail(FEM_ERR_STATE, "no FP32 copy of this level");
    DevBuf<float> xf(n), bf(n), df(n), yf(n);
    convert_kernel<double, float><<<grid_for(n, 256), 256, 0, s>>>(n, x, xf.get());
    convert_kernel<double, float><<<grid_for(n, 256), 256, 0, s>>>(n, b, bf.get());
    convert_kernel<double, float><<<grid_for(n, 256), 256, 0, s>>>(n, d, df.get());
    HIP_LAUNCH_CHECK();
    smoother_step_t<float>(h, A, L.dinv32.get(), mode, c1, c2, xf.get(), bf.get(), df.get(), yf.get());
    convert_kernel<float, double><<<grid_for(n, 256), 256, 0, s>>>(n, yf.get(), y);
    convert_kernel<float, double><<<grid_for(n, 256), 256, 0, s>>>(n, df.get(), d);
    HIP_LAUNCH_CHECK();
    HIP_CHECK(hipStreamSynchronize(s));
  }
}

void apply_level_int(Handle& h, int lvl, int which, const double* x, double* y) {
  hipStream_t s = h.stream;
  if (which == 3) {
    // the coarsest-level solve the V-cycle applies (FP64 inverse in every
    // precision; b and x in the level's vector type)
    const Hierarchy& H = h.H;
    if (lvl != H.coarse) fail(FEM_ERR_ARG, "which 3 (coarse solve) needs the coarsest level");
    const int64_t nc = H.nc;
    if (H.precision == 0) {
      coarse_kernel<double><<<(unsigned)nc, 64, 0, s>>>(nc, 1, H.cinv64.get(), x, y);
      HIP_LAUNCH_CHECK();
    } else {
      DevBuf<float> bf(nc), xf(nc);
      convert_kernel<double, float><<<grid_for(nc, 256), 256, 0, s>>>(nc, x, bf.get());
      coarse_kernel<float><<<(unsigned)nc, 64, 0, s>>>(nc, 1, H.cinv64.get(), bf.get(), xf.get());
      convert_kernel<float, double><<<grid_for(nc, 256), 256, 0, s>>>(nc, xf.get(), y);
      HIP_LAUNCH_CHECK();
      HIP_CHECK(hipStreamSynchronize(s));
    }
    return;
  }
  const Csr& M = level_matrix_of(h, lvl, which);
  if (h.H.precision == 0) {
    spmv_op<double, kAssign>(M, 1, x, y, nullptr, (const double*)nullptr, nullptr, nullptr, 0.0, 0.0, s);
  } else {
    if (!M.v32.size() || (M.nslices > 0 && !M.s32.size())) fail(FEM_ERR_STATE, "no FP32 copy of this matrix");
    DevBuf<float> xf(M.m > 0 ? M.m : 1), yf(M.n > 0 ? M.n : 1);
    if (M.m > 0) {
      convert_kernel<double, float><<<grid_for(M.m, 256), 256, 0, s>>>(M.m, x, xf.get());
      HIP_LAUNCH_CHECK();
    }
    spmv_op<float, kAssign>(M, 1, xf.get(), yf.get(), nullptr, (const float*)nullptr, nullptr, nullptr, 0.0f, 0.0f, s);
    if (M.n > 0) {
      convert_kernel<float, double><<<grid_for(M.n, 256), 256, 0, s>>>(M.n, yf.get(), y);
      HIP_LAUNCH_CHECK();
    }
    HIP_CHECK(hipStreamSynchronize(s));
  }
}

int padded_columns(int k, bool fp64) {
  // whole 16-byte groups: pairs in FP64, fours where FP32 vectors take part.
  // Kernels for any count had a lane per column and walked the coarse levels'
  // long rows serially (43 us for 832 rows).  An iteration of theirs, of fours
  // in every precision, and of this rule: 161^3 FP64, 2 columns 4.55, 3.60 and
  // 1.96 ms, 6 columns 5.71, 4.40 and 4.04; 1003 x 701 FP64, 6 columns 626, 713
  // and 577 us; 161^3 mixed, 2 columns 3.36 and 1.84 ms, 5 columns 5.14 and 2.9.
  if (k <= 1) return 1;
  const int g = fp64 ? 2 : 4;
  return (k + g - 1) / g * g;
}

void ensure_krylov(Handle& h, int k) {
  const int64_t n = h.A.n;
  if (k > 1) {
    // staging lists of blocks of kMultiSlices slices beside the one-column
    // lists of larger blocks (whose x rows do not fit LDS two blocks a CU)
    auto lists = [&](Csr& A) {
      if (A.nslices > 0 && A.sell_g == 1 && A.lds.bs > kMultiSlices && A.ldm.bs == 0)
        build_lds(A, kMultiSlices, A.ldm, h.stream);
    };
    lists(h.A);
    for (auto& Lp : h.H.levels) {
      lists(Lp->A);
    }
  }
  if (h.kcap < k) {
    ++h.gen;
    h.kcap = 0;  // until all are there: an allocation that fails leaves some empty
    h.kx.resize(n * k); h.kr.resize(n * k); h.kp.resize(n * k); h.kq.resize(n * k);
    h.kz.resize(n * k); h.kb.resize(n * k);
    h.ubuf.resize(n * k); h.ubuf2.resize(n * k);
    h.partials.resize((size_t)std::max<int64_t>(4096, n / 128 + 2) * 64);
    h.scal.resize((size_t)S_COUNT * 64);
    if (!h.h_scal) HIP_CHECK(hipHostMalloc((void**)&h.h_scal, sizeof(double) * S_COUNT * 64, hipHostMallocDefault));
    if (!h.h_act) {
      HIP_CHECK(hipHostMalloc((void**)&h.h_act, sizeof(double) * 2 * kActRec,
                              hipHostMallocMapped | hipHostMallocCoherent));
      HIP_CHECK(hipHostGetDevicePointer((void**)&h.d_act, h.h_act, 0));
    }
    h.kcap = k;
  }
  for (auto& Lp : h.H.levels) {
    Level& L = *Lp;
    if (L.wk >= k) continue;
    ++h.gen;
    L.wk = 0;
    const int64_t nl = (&L == h.H.levels[0].get()) ? h.A.n : L.A.n;
    if (h.H.precision == 0) {
      L.x64.resize(nl * k); L.t64.resize(nl * k); L.b64.resize(nl * k); L.r64.resize(nl * k); L.d64.resize(nl * k);
    } else {
      L.x32.resize(nl * k); L.t32.resize(nl * k); L.b32.resize(nl * k); L.r32.resize(nl * k); L.d32.resize(nl * k);
    }
    L.wk = k;
  }
}

// the preconditioner as PCG applies it (for one column: the fused level-0 ends
// and, in precision 2, the FP16 level-0 smoother; the r.z partials are unused)
void apply_vcycle_fp64(Handle& h, const double* r, double* z) { precondition(h, r, z, 1, h.partials.get()); }

namespace {

// Runs `body` (a fixed sequence of launches on h.stream that reads and writes
// device memory only) either directly or as a HIP graph captured at its first
// use and replayed while the buffers, hierarchy, k and tolerance it was
// captured with are unchanged.  Replays launch the same kernels with the same
// arguments, so results are bitwise those of the direct launches.
template <typename Fn>
void run_iteration(Handle& h, int k, double tol2, Fn&& body) {
  if (h.prm.launchMode == 0 || h.profiling || h.stream == nullptr) {
    body();
    return;
  }
  if (h.iter_graph && (h.graph_gen != h.gen || h.graph_k != k || h.graph_tol2 != tol2)) {
    HIP_CHECK(hipGraphExecDestroy(h.iter_graph));
    h.iter_graph = nullptr;
  }
  if (!h.iter_graph) {
    HIP_CHECK(hipStreamBeginCapture(h.stream, hipStreamCaptureModeRelaxed));
    try {
      body();
    } catch (...) {
      hipGraph_t junk = nullptr;
      (void)hipStreamEndCapture(h.stream, &junk);
      if (junk) (void)hipGraphDestroy(junk);
      throw;
    }
    hipGraph_t g = nullptr;
    HIP_CHECK(hipStreamEndCapture(h.stream, &g));
    hipError_t e = hipGraphInstantiate(&h.iter_graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    HIP_CHECK(e);
    h.graph_gen = h.gen;
    h.graph_k = k;
    h.graph_tol2 = tol2;
  }
  HIP_CHECK(hipGraphLaunch(h.iter_graph, h.stream));
}

void finish(Handle& h, int nb, int k, int mode, int slot, double tol2 = 0.0, int64_t at = 0) {
  pcg_finish_kernel<<<(unsigned)k, kFinNT, 0, h.stream>>>(nb, k, h.partials.get() + at, h.scal.get(), mode, slot, tol2,
                                                 mode == F_RR ? h.d_act : nullptr);
  HIP_LAUNCH_CHECK();
}

template <int KP, typename B>
unsigned launch_dot(Handle& h, int k, const double* a, const B* b) {
  const int64_t n = h.A.n;
  unsigned g = vec_grid(n, KP);
  pcg_dot_kernel<KP, B><<<g, kNT, 0, h.stream>>>(n, k, a, b, h.partials.get());
  HIP_LAUNCH_CHECK();
  return g;
}

// partials of a.b; returns their count per column
template <typename B>
unsigned dot_partials(Handle& h, int k, const double* a, const B* b) {
  switch (pow2_at_least(k)) {
    case 1: return launch_dot<1, B>(h, k, a, b);
    case 2: return launch_dot<2, B>(h, k, a, b);
    case 4: return launch_dot<4, B>(h, k, a, b);
    case 8: return launch_dot<8, B>(h, k, a, b);
    case 16: return launch_dot<16, B>(h, k, a, b);
    case 32: return launch_dot<32, B>(h, k, a, b);
    default: return launch_dot<64, B>(h, k, a, b);
  }
}

// mode F_STORE: scal[slot] = a.b; F_BETA: beta = a.b / rz, rz = a.b
template <typename B>
void dot(Handle& h, int k, const double* a, const B* b, int mode, int slot) {
  finish(h, (int)dot_partials(h, k, a, b), k, mode, slot);
}

// whether the kernel that reads alpha or beta sums the nb partials itself
bool folds(const Handle& h, int k, unsigned nb) { return k == 1 && h.A.n <= kFoldRows && nb <= (unsigned)kFoldParts; }

template <int KP, typename T>
void launch_update(Handle& h, int k, double tol2, const First0<T>& f0, unsigned npq, int rz) {
  const int64_t n = h.A.n;
  unsigned g = vec_grid(n, KP);
  const bool fold = folds(h, k, npq);
  if (!fold) finish(h, (int)npq, k, F_ALPHA, rz);
  // its own partials past those that its blocks read
  const int64_t at = fold ? kFoldParts : 0;
  auto go = [&](auto f) {
    pcg_update_kernel<KP, T, f.value><<<g, kNT, 0, h.stream>>>(
        n, k, h.kx.get(), h.kr.get(), h.kp.get(), h.kq.get(), h.partials.get() + at, h.scal.get(), f0.b, f0.dinv,
        f0.x0, f0.d0, f0.c0, h.partials.get(), (int)npq, rz, h.scal.get());
  };
  if constexpr (KP == 1) {
    if (fold) go(std::true_type{});
    else go(std::false_type{});
  } else {
    go(std::false_type{});
  }
  HIP_LAUNCH_CHECK();
  finish(h, (int)g, k, F_RR, rz, tol2, at);
}

// x += alpha p, r -= alpha q, |r|^2, and what f0 names: fl32(r) into the
// level-0 right-hand side, the smoother's first step from zero into its x and d;
// alpha from the npq partials of p.q and r.z in slot rz
template <typename T>
void update(Handle& h, int k, double tol2, const First0<T>& f0, unsigned npq, int rz) {
  switch (pow2_at_least(k)) {
    case 1: launch_update<1, T>(h, k, tol2, f0, npq, rz); break;
    case 2: launch_update<2, T>(h, k, tol2, f0, npq, rz); break;
    case 4: launch_update<4, T>(h, k, tol2, f0, npq, rz); break;
    case 8: launch_update<8, T>(h, k, tol2, f0, npq, rz); break;
    case 16: launch_update<16, T>(h, k, tol2, f0, npq, rz); break;
    case 32: launch_update<32, T>(h, k, tol2, f0, npq, rz); break;
    default: launch_update<64, T>(h, k, tol2, f0, npq, rz); break;
  }
}

unsigned launch_sell_dot(Handle& h) {
  const Csr& A = h.A;
  if (A.srow.size() || A.sell_g != 1)
    fail(FEM_ERR_STATE, "the operator's sliced-ELL copy must keep the row order with one lane per row");
  if (A.lds.bs > 0) {
    unsigned blocks = 0;
    lds_launch(A, 8, [&](auto head, unsigned nb, unsigned nt) {
      pcg_sell_lds_dot_kernel<head.value><<<nb, nt, sizeof(double) * (size_t)A.lds.maxc, h.stream>>>(
          A.n, A.nslices, sell_view(A), lds_view(A.lds), A.s64.get(), h.kp.get(), h.kq.get(), h.partials.get());
      blocks = nb;
    });
    HIP_LAUNCH_CHECK();
    return blocks;
  }
  unsigned g = grid_for(A.nslices, kNT / 64);
  pcg_sell_dot_kernel<<<g, kNT, 0, h.stream>>>(A.n, A.nslices, sell_view(A), A.s64.get(), h.kp.get(), h.kq.get(),
                                               h.partials.get());
  HIP_LAUNCH_CHECK();
  return (unsigned)g;
}

template <int G>
unsigned launch_spmv_dot(Handle& h) {
  const Csr& A = h.A;
  int64_t g = (A.n * G + kNT - 1) / kNT;
  if (g > 4096) g = 4096;
  pcg_spmv_dot_kernel<G><<<(unsigned)g, kNT, 0, h.stream>>>(A.n, A.rp.get(), A.ci.get(), A.v64.get(), h.kp.get(),
                                                            h.kq.get(), h.partials.get());
  HIP_LAUNCH_CHECK();
  return (unsigned)g;
}

template <int L>
unsigned launch_spmm_dot(Handle& h, int k) {
  const Csr& A = h.A;
  int64_t g = (A.n * L + kNT - 1) / kNT;
  if (g > 4096) g = 4096;
  pcg_spmm_dot_vec_kernel<L><<<(unsigned)g, kNT, 0, h.stream>>>(A.n, k, A.rp.get(), A.ci.get(), A.v64.get(), h.kp.get(),
                                                                h.kq.get(), h.partials.get());
  HIP_LAUNCH_CHECK();
  return (unsigned)g;
}

// q = A p; returns the count of p.q partials per column
unsigned spmv_dot(Handle& h, int k) {
  const Csr& A = h.A;
  ProfScope ps(h, "pcg_spmv", matrix_bytes<double>(A, k) + 3.0 * 8 * A.n * k);
  if (k == 1 && A.nslices > 0 && A.s64.size() && A.sell_g == 1 && A.srow.size() == 0) {
    return launch_sell_dot(h);
  } else if (k == 1) {
    switch (lanes_for(A)) {
      case 4: return launch_spmv_dot<4>(h);
      case 8: return launch_spmv_dot<8>(h);
      case 16: return launch_spmv_dot<16>(h);
      case 32: return launch_spmv_dot<32>(h);
      default: return launch_spmv_dot<64>(h);
    }
  } else if (multi_staged<double>(A, k) && A.srow.size() == 0) {
    launch_lds_multi<double, kAssign, 1>(A, k, h.kp.get(), h.kq.get(), nullptr, (const double*)nullptr, nullptr,
                                         nullptr, 0.0, 0.0, nullptr, h.partials.get(), h.stream);
    HIP_LAUNCH_CHECK();
    return multi_blocks(A);
  } else {
    switch (pow2_at_least(k / 2)) {
      case 1: return launch_spmm_dot<1>(h, k);
      case 2: return launch_spmm_dot<2>(h, k);
      case 4: return launch_spmm_dot<4>(h, k);
      case 8: return launch_spmm_dot<8>(h, k);
      case 16: return launch_spmm_dot<16>(h, k);
      default: return launch_spmm_dot<32>(h, k);
    }
  }
}

void set_scal(Handle& h, int slot, int k, const double* v) {
  HIP_CHECK(hipMemcpyAsync(h.scal.get() + slot * k, v, sizeof(double) * k, hipMemcpyHostToDevice, h.stream));
}

// Convergence record `seq` of the |r|^2 finish (act flags and |r|^2 per
// column), read from host-mapped memory once event `ev` (recorded after that
// finish) has completed; polled, so there is no sleep / wake-up in between.
void read_record(Handle& h, hipEvent_t ev, uint64_t seq, int k, double* act, double* rr) {
  for (;;) {
    const hipError_t e = hipEventQuery(ev);
    if (e == hipSuccess) break;
    if (e != hipErrorNotReady) HIP_CHECK(e);
  }
  const volatile double* rec = h.h_act + (seq & 1) * kActRec;
  if (rec[128] != (double)seq) fail(FEM_ERR_STATE, "convergence record out of sequence");
  for (int c = 0; c < k; ++c) {
    act[c] = rec[c];
    rr[c] = rec[64 + c];
  }
}

void get_scal(Handle& h, int slot, int k, double* v) {
  HIP_CHECK(hipMemcpyAsync(h.h_scal, h.scal.get() + slot * k, sizeof(double) * k, hipMemcpyDeviceToHost, h.stream));
  HIP_CHECK(hipStreamSynchronize(h.stream));
  std::memcpy(v, h.h_scal, sizeof(double) * k);
}

}  // namespace

// Solve A x = b for k columns held in h.kb / h.kx (internal numbering).
int pcg_solve(Handle& h, int k, fem_solve_info* info) {
  hipStream_t s = h.stream;
  const int64_t n = h.A.n;
  const int64_t m = n * k;
  const double tol = h.prm.tolerance;
  const double tol2 = tol * tol;
  std::vector<double> bb(k), rr(k), act(k), one(k, 1.0);

  hipEvent_t e0, e1;
  HIP_CHECK(hipEventCreate(&e0));
  HIP_CHECK(hipEventCreate(&e1));
  HIP_CHECK(hipEventRecord(e0, s));

  dot(h, k, h.kb.get(), h.kb.get(), F_STORE, S_BB);
  get_scal(h, S_BB, k, bb.data());

  int iters = 0;
  int status = FEM_OK;
  auto true_residual = [&](std::vector<double>& rel) {
    // kq = b - A x ; rel_c = ||kq_c|| / ||b_c||
    spmv_op<double, kResid>(h.A, k, h.kx.get(), h.kq.get(), h.kb.get(), (const double*)nullptr, nullptr, nullptr,
                            0.0, 0.0, s);
    dot(h, k, h.kq.get(), h.kq.get(), F_STORE, S_TRUE);
    std::vector<double> t(k);
    get_scal(h, S_TRUE, k, t.data());
    rel.resize(k);
    for (int c = 0; c < k; ++c) rel[c] = bb[c] > 0 ? std::sqrt(t[c] / bb[c]) : 0.0;
  };

  std::vector<double> rel(k, 0.0);
  if (h.prm.solverType == 0) {
    // one V-cycle: x = M b (the initial guess is not used, as in the reference)
    precondition(h, h.kb.get(), h.kx.get(), k);
    iters = 1;
    true_residual(rel);
    for (int c = 0; c < k; ++c)
      if (rel[c] > tol) status = FEM_ERR_NOT_CONVERGED;
  } else {
    // a zero right-hand side has the exact solution x = 0, whatever the
    // initial guess (its column then starts, and stays, converged)
    unsigned long long zmask = 0;
    for (int c = 0; c < k; ++c)
      if (!(bb[c] > 0)) zmask |= 1ull << c;
    if (zmask) {
      zero_cols_kernel<<<grid_for(m, 256), 256, 0, s>>>(m, k, zmask, h.kx.get());
      HIP_LAUNCH_CHECK();
    }
    // r = b - A x0
    spmv_op<double, kResid>(h.A, k, h.kx.get(), h.kr.get(), h.kb.get(), (const double*)nullptr, nullptr, nullptr,
                            0.0, 0.0, s);
    dot(h, k, h.kr.get(), h.kr.get(), F_STORE, S_RR);
    get_scal(h, S_RR, k, rr.data());
    bool any = false;
    for (int c = 0; c < k; ++c) {
      act[c] = (bb[c] > 0 && rr[c] > tol2 * bb[c]) ? 1.0 : 0.0;
      any = any || act[c] != 0.0;
    }
    set_scal(h, S_ACT, k, act.data());
    const std::vector<double> zero_seq(k, 0.0);
    set_scal(h, S_SEQ, k, zero_seq.data());  // |r|^2 finishes of this solve are numbered from 1
    uint64_t seq_issued = 0;
    bool ahead = false;
    hipEvent_t evs[2];
    HIP_CHECK(hipEventCreateWithFlags(&evs[0], hipEventDisableTiming));
    HIP_CHECK(hipEventCreateWithFlags(&evs[1], hipEventDisableTiming));
    struct EvGuard {
      hipEvent_t* e;
      ~EvGuard() {
        (void)hipEventDestroy(e[0]);
        (void)hipEventDestroy(e[1]);
      }
    } ev_guard{evs};
    int restarts = 0;
    // the level-0 smoother's first step from zero (on fl32(r) in the mixed
    // precisions) comes from the update; an unfused mixed-precision V-cycle
    // without one still takes fl32(r)
    First0<float> f32 = first0_for<float>(h, k);
    const First0<double> f64 = first0_for<double>(h, k);
    if (!f32.on && h.H.precision >= 1 && !fused_level0(h, k, true)) f32.b = h.H.levels[0]->b32.get();
    auto operator_update = [&](int rz) {  // q = A p, alpha; x, r, rr, act
      const unsigned npq = spmv_dot(h, k);
      if (f64.on) update<double>(h, k, tol2, f64, npq, rz);
      else update<float>(h, k, tol2, f32, npq, rz);
    };
    while (any) {
      // z = M r and partials of r.z (fused into the last level-0 smoothing step
      // when possible); z stays where the preconditioner left it
      auto precondition_dot = [&](bool r32_ready) {
        PrecOut o = precondition_pcg(h, h.kr.get(), h.kz.get(), k, h.partials.get(),
                                           r32_ready && f32.b, r32_ready && (f32.on || f64.on));
        if (!o.nb) o.nb = o.z32 ? dot_partials(h, k, h.kr.get(), o.z32) : dot_partials(h, k, h.kr.get(), o.z64);
        return o;
      };
      const PrecOut o0 = precondition_dot(false);
      finish(h, (int)o0.nb, k, F_STORE, S_RZ);
      if (o0.z32) convert_kernel<float, double><<<grid_for(m, 256), 256, 0, s>>>(m, o0.z32, h.kp.get());
      else copy_kernel<<<grid_for(m, 256), 256, 0, s>>>(m, o0.z64, h.kp.get());
      HIP_LAUNCH_CHECK();
      // the first iteration starts from p = z; every later one is the fixed
      // sequence below (captured once, then replayed), which follows an update
      // (so fl32(r) is in place)
      // an F-cycle is not a symmetric preconditioner: its beta is the flexible one
      const bool flexible = cycle_type(h) == kCycleF;
      auto iteration = [&]() {
        // z, beta, rz
        const PrecOut o = precondition_dot(true);
        if (!flexible && folds(h, k, o.nb)) {
          const unsigned g = grid_for(n, kNT);
          if (o.z32)
            pcg_p_fold_kernel<float><<<g, kNT, 0, s>>>(n, o.z32, h.kp.get(), h.scal.get(), h.partials.get(), (int)o.nb);
          else
            pcg_p_fold_kernel<double><<<g, kNT, 0, s>>>(n, o.z64, h.kp.get(), h.scal.get(), h.partials.get(),
                                                        (int)o.nb);
          HIP_LAUNCH_CHECK();
          operator_update(S_RZN);
          return;
        }
        finish(h, (int)o.nb, k, flexible ? F_STORE : F_BETA, flexible ? S_RZN : 0);
        if (flexible) {
          if (o.z32) dot(h, k, h.kq.get(), o.z32, F_FLEX, 0);
          else dot(h, k, h.kq.get(), o.z64, F_FLEX, 0);
        }
        if (o.z32)
          pcg_p_kernel<float><<<grid_for(m, 256), 256, 0, s>>>(m, k, o.z32, h.kp.get(), h.scal.get());
        else
          pcg_p_kernel<double><<<grid_for(m, 256), 256, 0, s>>>(m, k, o.z64, h.kp.get(), h.scal.get());
        HIP_LAUNCH_CHECK();
        operator_update(S_RZ);
      };
      // Iteration n ends with the n-th |r|^2 finish of this solve; the host
      // reads its record while iteration n + 1 may already run: the next
      // iteration is queued ahead whenever the residual history predicts
      // more than two further iterations.  An iteration queued after the
      // last needed one leaves x and r unchanged (alpha = beta = 0 for
      // converged columns).
      const uint64_t seq0 = seq_issued;
      auto issue = [&](bool first) {
        if (first) {
          operator_update(S_RZ);
        } else {
          run_iteration(h, k, tol2, iteration);
        }
        ++seq_issued;
        HIP_CHECK(hipEventRecord(evs[seq_issued & 1], s));
      };
      if (iters < h.prm.maxIters) issue(true);
      uint64_t seq_done = seq0;
      std::vector<double> rr_prev(k, -1.0), rr_prev2(k, -1.0), rrn(k);
      while (seq_done < seq_issued) {
        const bool room = iters + (int)(seq_issued - seq_done) < h.prm.maxIters;
        if (ahead && room && seq_issued == seq_done + 1) issue(false);
        read_record(h, evs[(seq_done + 1) & 1], seq_done + 1, k, act.data(), rrn.data());
        ++seq_done;
        ++iters;
        bool still = false;
        double remaining = 0.0;
        for (int c = 0; c < k; ++c) {
          if (act[c] == 0.0) continue;
          still = true;
          // iterations left at the geometric rate of the last two
          double rem = 1e30;
          if (rr_prev2[c] > 0.0 && rrn[c] > 0.0 && rrn[c] < rr_prev2[c])
            rem = std::log(tol2 * bb[c] / rrn[c]) / (0.5 * std::log(rrn[c] / rr_prev2[c]));
          remaining = std::max(remaining, rem);
          rr_prev2[c] = rr_prev[c];
          rr_prev[c] = rrn[c];
        }
        if (!still || iters >= h.prm.maxIters) break;
        ahead = remaining > 2.0;
        if (seq_issued == seq_done) issue(false);
      }
      // verify on the true residual; restart columns that drifted
      true_residual(rel);
      any = false;
      for (int c = 0; c < k; ++c) {
        act[c] = (rel[c] > tol) ? 1.0 : 0.0;
        any = any || act[c] != 0.0;
      }
      if (!any || iters >= h.prm.maxIters || restarts >= 3) break;
      ++restarts;
      copy_kernel<<<grid_for(m, 256), 256, 0, s>>>(m, h.kq.get(), h.kr.get());
      HIP_LAUNCH_CHECK();
      set_scal(h, S_ACT, k, act.data());
    }
    if (any) status = FEM_ERR_NOT_CONVERGED;
    if (rel.empty() || iters == 0) true_residual(rel);
    for (int c = 0; c < k; ++c)
      if (rel[c] > tol) status = FEM_ERR_NOT_CONVERGED;
  }
  HIP_CHECK(hipEventRecord(e1, s));
  HIP_CHECK(hipEventSynchronize(e1));
  float ms = 0.f;
  HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (info) {
    info->iterations = iters;
    double mx = 0.0;
    for (int c = 0; c < k; ++c) mx = std::max(mx, rel[c]);
    info->rel_residual = mx;
    info->converged = (status == FEM_OK) ? 1 : 0;
    info->solve_ms = ms;
  }
  return status;
}

// ---- allocation-free preconditioner application ---------------------------------
// Device scratch of apply_preconditioner_noalloc: r and z in internal
// numbering (kNoAllocRows doubles each), then the r.z partials of the fused
// level-0 smoother's last step (at most one per 64-row slice).  The array is
// one copy per GPU, held until the process ends, and shared by every call on
// that GPU.  Its name is a host-side stand-in in host code: kernels receive
// the per-device address from hipGetSymbolAddress.
constexpr int64_t kNoAllocRows = (int64_t)1 << 21;
constexpr int64_t kNoAllocPartials = kNoAllocRows / 64 + 64;
static __device__ __align__(256) double scratch[2 * kNoAllocRows + kNoAllocPartials];

namespace {
std::mutex g_scratch_mu;
std::map<int, double*> g_scratch_addr;  // device ordinal -> address of scratch

// the address of scratch on device dev, which must be the current device
// (looked up once per device)
double* scratch_address(int dev) {
  int cur = -1;
  HIP_CHECK(hipGetDevice(&cur));
  if (cur != dev)
    fail(FEM_ERR_STATE, "the current HIP device (" + std::to_string(cur) + ") is not the handle's device (" +
                            std::to_string(dev) + ")");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  auto it = g_scratch_addr.find(dev);
  if (it != g_scratch_addr.end()) return it->second;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || p == nullptr)
    fail(FEM_ERR_HIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
  g_scratch_addr[dev] = static_cast<double*>(p);
  return static_cast<double*>(p);
}
}  // namespace

int64_t noalloc_max_rows() { return kNoAllocRows; }

void noalloc_init(const Handle& h) {
  int cur = -1;
  if (hipGetDevice(&cur) == hipSuccess && cur == h.device) (void)scratch_address(h.device);
}

void apply_preconditioner_noalloc(Handle& h, const double* r_user, double* z_user) {
  const int64_t n = h.A.n;
  if (n == 0) fail(FEM_ERR_EMPTY, "Error no matrix specified");
  if (n > kNoAllocRows)
    fail(FEM_ERR_CAPACITY, "fem_apply_preconditioner_noalloc: " + std::to_string(n) +
                               " rows exceed its limit of " + std::to_string(kNoAllocRows) + " rows");
  if (!h.H.built) fail(FEM_ERR_STATE, "fem_apply_preconditioner_noalloc: no hierarchy; call fem_setup first");
  bool ready = h.kcap >= 1;
  for (auto& Lp : h.H.levels) ready = ready && Lp->wk >= 1;
  if (!ready) fail(FEM_ERR_STATE, "fem_apply_preconditioner_noalloc: work vectors missing; call fem_setup first");
  if (h.profiling) fail(FEM_ERR_STATE, "fem_apply_preconditioner_noalloc: profiling is enabled");
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  HIP_CHECK(hipStreamIsCapturing(h.stream, &cap));
  if (cap != hipStreamCaptureStatusNone) h.captured = true;
  double* base = scratch_address(h.device);
  double* r = base;
  double* z = base + kNoAllocRows;
  double* partials = base + 2 * kNoAllocRows;
  gather_user_to_int(h, r_user, r, 1, 1);
  precondition(h, r, z, 1, partials);
  scatter_int_to_user(h, z, z_user, 1, 1);
}

}  // namespace fem
