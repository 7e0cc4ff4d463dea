// lu.hip -- batched LU of the element matrices with partial pivoting, the solves with it, and the mixed
// form's refinement right-hand side (uequation.cpp:683-711's inverse of D' applied to F' and Ru).
#include "blkval.hpp"
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace exa {

namespace {

// f(0), f(1), .. with compile-time indices (register arrays indexed by them stay in registers, which
// an unroll pragma does not promise for long bodies)
template <int... I, typename F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>()), ...);
}

// ---------------------------------------------------------------------------
// Right-looking blocked LU of the augmented systems [D | RHS] (n x ncols, ld n),
// one panel of BLU_NB columns at a time: k_lu_panel factors the panel of every
// matrix in LDS (partial pivoting), swaps the rows of the columns right of the
// panel and solves L11 U12 = A12; the trailing update A22 -= L21 U12 and the
// back substitution's updates run on the MFMA GEMM.
// ---------------------------------------------------------------------------
constexpr int BLU_MIN_N = 64;  // smaller blocks use the single-kernel k_lu_small

template <typename T, int BLU_NB>
__global__ __launch_bounds__(256) void k_lu_panel(T* Aall, int n, int ncols, long stride, int k0,
                                                  int* info, int* pivout) {
  T* A = Aall + stride * blockIdx.x;
  const int nb = min(BLU_NB, n - k0);
  const int rows = n - k0;
  extern __shared__ double lu_sm[];
  T* P = reinterpret_cast<T*>(lu_sm);  // rows x nb, ld rows
  __shared__ double wv[4];
  __shared__ int wi[4];
  __shared__ int piv[BLU_NB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int idx = tid; idx < rows * nb; idx += 256) {
    int r = idx % rows, kk = idx / rows;
    P[idx] = A[k0 + r + static_cast<long>(n) * (k0 + kk)];
  }
  __syncthreads();
  int singular = 0;
  for (int kk = 0; kk < nb; ++kk) {
    double best = -1.0;
    int bi = kk;
    for (int r = kk + tid; r < rows; r += 256) {
      double v = fabs(P[r + rows * kk]);
      if (v > best) { best = v; bi = r; }
    }
    argmax_wave(best, bi);
    if (lane == 0) { wv[wave] = best; wi[wave] = bi; }
    __syncthreads();
    if (tid == 0) {
      double b = wv[0];
      int p = wi[0];
      for (int w = 1; w < 4; ++w)
        if (wv[w] > b || (wv[w] == b && wi[w] < p)) { b = wv[w]; p = wi[w]; }
      piv[kk] = p;
    }
    __syncthreads();
    const int p = piv[kk];
    if (p != kk && tid < nb) {
      T t = P[kk + rows * tid];
      P[kk + rows * tid] = P[p + rows * tid];
      P[p + rows * tid] = t;
    }
    __syncthreads();
    const T pv = P[kk + rows * kk];
    if (pv == 0.0) singular = 1;
    const T inv = T(1) / pv;
    for (int r = kk + 1 + tid; r < rows; r += 256) P[r + rows * kk] *= inv;
    __syncthreads();
    const int rr = rows - kk - 1, cc = nb - kk - 1;
    for (int idx = tid; idx < rr * cc; idx += 256) {
      int r = kk + 1 + idx % rr, c = kk + 1 + idx / rr;
      P[r + rows * c] = fma(-P[r + rows * kk], P[kk + rows * c], P[r + rows * c]);
    }
    __syncthreads();
  }
  for (int idx = tid; idx < rows * nb; idx += 256) {
    int r = idx % rows, kk = idx / rows;
    A[k0 + r + static_cast<long>(n) * (k0 + kk)] = P[idx];
  }
  // columns right of the panel: row swaps, then U12 = L11^{-1} A12
  for (int j = k0 + nb + tid; j < ncols; j += 256) {
    T* colj = A + static_cast<long>(n) * j + k0;
    T x[BLU_NB];
#pragma unroll
    for (int kk = 0; kk < BLU_NB; ++kk) x[kk] = (kk < nb) ? colj[kk] : 0.0;
    // pivots are applied in order; p < BLU_NB means both rows are in the register
    // block (a last panel narrower than BLU_NB has rows == nb)
#pragma unroll
    for (int kk = 0; kk < BLU_NB; ++kk) {
      if (kk < nb) {
        const int p = piv[kk];
        if (p != kk) {
          if (p < BLU_NB) {
#pragma unroll
            for (int q = kk + 1; q < BLU_NB; ++q)
              if (q == p) {
                const T t = x[q];
                x[q] = x[kk];
                x[kk] = t;
              }
          } else {
            const T t = colj[p];
            colj[p] = x[kk];
            x[kk] = t;
          }
        }
      }
    }
#pragma unroll
    for (int kk = 1; kk < BLU_NB; ++kk)
#pragma unroll
      for (int t = 0; t < kk; ++t)
        if (kk < nb) x[kk] = fma(-P[kk + rows * t], x[t], x[kk]);
#pragma unroll
    for (int kk = 0; kk < BLU_NB; ++kk)
      if (kk < nb) colj[kk] = x[kk];
  }
  if (tid == 0 && info) info[blockIdx.x] = (k0 == 0 ? 0 : info[blockIdx.x]) | singular;
  // panel-relative pivots of this panel (row k0+kk was exchanged with row k0+piv[kk])
  if (pivout && tid < nb) pivout[static_cast<long>(blockIdx.x) * n + k0 + tid] = piv[tid];
}

// Lane 63 of a reduction over the wave by data-parallel moves: step CTRL takes another lane's (v, p) where
// the move reaches this lane (rows of RM), its own otherwise, and keeps the larger value, of equal ones the
// smaller index.
template <int CTRL, int RM>
__device__ __forceinline__ void argmax_step(double& v, int& p) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  const double ov = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, RM, 0xf, false),
                                     __builtin_amdgcn_update_dpp(lo, lo, CTRL, RM, 0xf, false));
  const int op = __builtin_amdgcn_update_dpp(p, p, CTRL, RM, 0xf, false);
  if (ov > v || (ov == v && op < p)) {
    v = ov;
    p = op;
  }
}
template <int CTRL, int RM>
__device__ __forceinline__ void argmax_step(float& v, int& p) {
  const int b = __float_as_int(v);
  const float ov = __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, RM, 0xf, false));
  const int op = __builtin_amdgcn_update_dpp(p, p, CTRL, RM, 0xf, false);
  if (ov > v || (ov == v && op < p)) {
    v = ov;
    p = op;
  }
}
// the index of the wave's largest value (of equal ones the smallest index), to every lane
template <typename T>
__device__ __forceinline__ int argmax_lanes(T v, int p) {
  argmax_step<0x111, 0xf>(v, p);  // row_shr:1
  argmax_step<0x112, 0xf>(v, p);  // row_shr:2
  argmax_step<0x114, 0xf>(v, p);  // row_shr:4
  argmax_step<0x118, 0xf>(v, p);  // row_shr:8
  argmax_step<0x142, 0xa>(v, p);  // row_bcast:15
  argmax_step<0x143, 0xc>(v, p);  // row_bcast:31
  return __builtin_amdgcn_readlane(p, 63);
}
__device__ __forceinline__ double lane_value(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The panel factorisation of k_lu_panel with one wave per matrix, for panels of at most 256 rows: lane t
// holds rows t, t + 64, .. (RPL of them) of the rows x nb panel in registers.  No row moves: each row
// keeps its position pos in the exchanged order (pivots are chosen among pos >= kk, ties to the smaller),
// the pivot row reaches every lane through scalar registers, and rows are written to their positions at
// the end.  A column's chain is the argmax, the broadcast, one reciprocal and the update, without a
// barrier, and a SIMD runs the chains of its waves side by side.  The operations on every entry are those
// of k_lu_panel, so the factors are the same.  piv_ws + blockIdx.x*pws: the number of rows that moved, then
// (new, old) row of each, for the columns right of the panel.  Per launch, against a workgroup of four waves per
// matrix with two barriers per column: 2025 FP64 matrices of up to 144 rows, 32 columns 156 -> 53 us; 2667 of up
// to 250 rows 200 us -> 112 us; 4096 FP32 matrices of 100 rows, 64 columns 484 -> 190 us.
template <typename T, int NB, int RPL>
__global__ __launch_bounds__(64) void k_lu_panel_wave(T* Aall, int n, long stride, int k0, int* info, int* pivout,
                                                      int* piv_ws, int pws) {
  T* A = Aall + stride * blockIdx.x + k0 + static_cast<long>(n) * k0;
  const int nb = min(NB, n - k0);
  const int rows = n - k0;  // <= 64 RPL
  const int lane = threadIdx.x;
  T a[RPL][NB];
  int pos[RPL];
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    const int r = lane + 64 * q;
    pos[q] = r < rows ? r : -1;
#pragma unroll
    for (int c = 0; c < NB; ++c) a[q][c] = (r < rows && c < nb) ? A[r + static_cast<long>(n) * c] : T(0);
  }
  int singular = 0;
  static_for(std::make_integer_sequence<int, NB>(), [&](auto KK) __attribute__((always_inline)) {
    constexpr int kk = decltype(KK)::value;
    if (kk < nb) {
      // (a column without a comparable entry, all NaN, keeps its row)
      T bv = T(-1);
      int bp = kk;
#pragma unroll
      for (int q = 0; q < RPL; ++q) {
        const T v = fabs(a[q][kk]);
        if (pos[q] >= kk && (v > bv || (v == bv && pos[q] < bp))) {
          bv = v;
          bp = pos[q];
        }
      }
      const int p = argmax_lanes(bv, bp);
      if (pivout && lane == 0) pivout[static_cast<long>(blockIdx.x) * n + k0 + kk] = p;
      T pr[NB];
#pragma unroll
      for (int q = 0; q < RPL; ++q) {
        const unsigned long long at = __ballot(pos[q] == p);
        if (at) {
          const int l = __builtin_ctzll(at);
#pragma unroll
          for (int c = kk; c < NB; ++c) pr[c] = lane_value(a[q][c], l);
        }
      }
      if (pr[kk] == T(0)) singular = 1;
      const T inv = T(1) / pr[kk];
#pragma unroll
      for (int q = 0; q < RPL; ++q) {
        pos[q] = pos[q] == p ? kk : pos[q] == kk ? p : pos[q];
        if (pos[q] > kk) {
          const T l = a[q][kk] * inv;
          a[q][kk] = l;
#pragma unroll
          for (int c = kk + 1; c < NB; ++c) a[q][c] = fma(-l, pr[c], a[q][c]);
        }
      }
    }
  });
  int* ws = piv_ws + static_cast<long>(blockIdx.x) * pws;
  int moved = 0;
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    const int r = lane + 64 * q;
    const bool mv = pos[q] >= 0 && pos[q] != r;
    const unsigned long long m = __ballot(mv);
    if (mv) {
      const int k = moved + __popcll(m & ((1ull << lane) - 1ull));
      ws[1 + 2 * k] = pos[q];
      ws[2 + 2 * k] = r;
    }
    moved += __popcll(m);
    if (pos[q] >= 0)
#pragma unroll
      for (int c = 0; c < NB; ++c)
        if (c < nb) A[pos[q] + static_cast<long>(n) * c] = a[q][c];
  }
  if (lane == 0) {
    ws[0] = moved;
    if (info) info[blockIdx.x] = (k0 == 0 ? 0 : info[blockIdx.x]) | singular;
  }
}

// The row exchanges of a panel factored by k_lu_panel_wave, applied to the columns right of it.  A wave
// takes 8 columns at a time, lane t the t-th moved row (and the t+64th): a column's rows lie in a few
// cache lines, which all lanes then share, where a lane per column touched a line per row and lane (n = 100,
// 4096 FP32 matrices: 52 us against 249; n = 144, 2025 FP64 matrices 46 us against 111).  All of a column's values are read before any is written.
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_lu_swap(T* Aall, int n, int ncols, long stride, int k0, const int* piv_ws,
                                                 int pws) {
  constexpr int SL = (2 * NB + 63) / 64;
  const int* ws = piv_ws + static_cast<long>(blockIdx.x) * pws;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nm = ws[0];
  const int first = k0 + min(NB, n - k0) + blockIdx.y * 64 + 16 * wave;
  T* A = Aall + stride * blockIdx.x + k0;
  int dst[SL], src[SL];
#pragma unroll
  for (int q = 0; q < SL; ++q) {
    const int i = lane + 64 * q;
    dst[q] = i < nm ? ws[1 + 2 * i] : 0;
    src[q] = i < nm ? ws[2 + 2 * i] : 0;
  }
  for (int j0 = first; j0 < min(first + 16, ncols); j0 += 8) {
    T v[8][SL];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int q = 0; q < SL; ++q)
        v[u][q] = A[src[q] + static_cast<long>(n) * min(j0 + u, ncols - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (j0 + u < ncols)
#pragma unroll
        for (int q = 0; q < SL; ++q)
          if (lane + 64 * q < nm) A[dst[q] + static_cast<long>(n) * (j0 + u)] = v[u][q];
  }
}

// Columns right of a panel factored by k_lu_panel_wave, after k_lu_swap: U12 = L11^{-1} A12 (one
// column per thread; blockIdx.y selects a chunk of 256 columns).  Each thread reads its column's
// nb contiguous entries; a variant with one wave per 64 columns staged through LDS with coalesced
// loads was measured slower (0.47 against 0.33 ms per launch, averaged over the FP64 LUs of the
// 32^3, p = 4 mesh's set-up and assembly; k_lu_back 0.31 against 0.26 ms): the LDS tile cut
// occupancy.
template <typename T, int BLU_NB>
__global__ __launch_bounds__(256) void k_lu_u12(T* Aall, int n, int ncols, long stride, int k0) {
  T* A = Aall + stride * blockIdx.x;
  const int nb = min(BLU_NB, n - k0);
  // L11 with a run-time leading dimension: constant LDS addresses in the unrolled solve let the
  // compiler hoist every load into registers (and spill)
  __shared__ T L11[BLU_NB * BLU_NB];
  const int ldl = nb;
  const int tid = threadIdx.x;
  for (int idx = tid; idx < nb * nb; idx += 256) {
    const int r = idx % nb, c = idx / nb;
    L11[r + ldl * c] = A[k0 + r + static_cast<long>(n) * (k0 + c)];
  }
  __syncthreads();
  const int j = k0 + nb + blockIdx.y * 256 + tid;
  if (j >= ncols) return;
  T* colj = A + static_cast<long>(n) * j + k0;
  T x[BLU_NB];
#pragma unroll
  for (int kk = 0; kk < BLU_NB; ++kk) x[kk] = (kk < nb) ? colj[kk] : 0.0;
#pragma unroll
  for (int kk = 1; kk < BLU_NB; ++kk)
#pragma unroll
    for (int t = 0; t < kk; ++t)
      if (kk < nb) x[kk] = fma(-L11[kk + ldl * t], x[t], x[kk]);
#pragma unroll
  for (int kk = 0; kk < BLU_NB; ++kk)
    if (kk < nb) colj[kk] = x[kk];
}

// Inverse of the unit lower triangle L11 (LOWER) or of the upper triangle U11 of the panel at
// k0, one workgroup per matrix: thread c computes column c by substitution (static register
// indices, predicated on c), written to W[blockIdx.x] (nb x nb, ld BLU_NB).  U12 = L11^{-1} A12
// and X = U11^{-1} X then run as in-place GEMMs on the matrix cores: each output tile covers all
// nb rows of its own columns, so it reads its B columns completely before writing them.
template <typename T, int BLU_NB, bool LOWER>
__global__ __launch_bounds__(64) void k_lu_tri_inv(const T* Aall, int n, long stride, int k0, T* W) {
  const T* A = Aall + stride * blockIdx.x;
  const int nb = min(BLU_NB, n - k0);
  __shared__ T Ts[BLU_NB][BLU_NB + 1];
  for (int idx = threadIdx.x; idx < nb * nb; idx += 64) {
    const int r = idx % nb, c = idx / nb;
    Ts[r][c] = A[k0 + r + static_cast<long>(n) * (k0 + c)];
  }
  __syncthreads();
  const int c = threadIdx.x;
  if (c >= nb) return;
  T y[BLU_NB];
  if (LOWER) {
#pragma unroll
    for (int r = 0; r < BLU_NB; ++r) {
      if (r <= c || r >= nb) {
        y[r] = (r == c) ? T(1) : T(0);
      } else {
        T s = T(0);
#pragma unroll
        for (int t = 0; t < r; ++t)
          if (t >= c) s = fma(Ts[r][t], y[t], s);
        y[r] = -s;
      }
    }
  } else {
#pragma unroll
    for (int r = BLU_NB - 1; r >= 0; --r) {
      if (r > c || r >= nb) {
        y[r] = T(0);
      } else if (r == c) {
        y[r] = T(1) / Ts[r][r];
      } else {
        T s = T(0);
#pragma unroll
        for (int t = r + 1; t < BLU_NB; ++t)
          if (t <= c) s = fma(Ts[r][t], y[t], s);
        y[r] = -s / Ts[r][r];
      }
    }
  }
  T* Wm = W + static_cast<long>(blockIdx.x) * BLU_NB * BLU_NB;
#pragma unroll
  for (int r = 0; r < BLU_NB; ++r)
    if (r < nb) Wm[r + BLU_NB * c] = y[r];
}

// X[k0:k0+nb, c] = U11^{-1} X[k0:k0+nb, c] for the right-hand-side columns c >= n
template <typename T, int BLU_NB>
__global__ __launch_bounds__(256) void k_lu_back(T* Aall, int n, int ncols, long stride, int k0) {
  T* A = Aall + stride * blockIdx.x;
  const int nb = min(BLU_NB, n - k0);
  __shared__ T U[BLU_NB][BLU_NB + 1];
  __shared__ T dinv[BLU_NB];
  const int tid = threadIdx.x;
  for (int idx = tid; idx < nb * nb; idx += 256) {
    int r = idx % nb, c = idx / nb;
    U[r][c] = A[k0 + r + static_cast<long>(n) * (k0 + c)];
  }
  __syncthreads();
  if (tid < nb) dinv[tid] = T(1) / U[tid][tid];
  __syncthreads();
  // one right-hand-side column per thread (blockIdx.y selects a chunk of 256)
  const int j = n + blockIdx.y * 256 + tid;
  if (j >= ncols) return;
  T* colj = A + static_cast<long>(n) * j + k0;
  T x[BLU_NB];
#pragma unroll
  for (int kk = 0; kk < BLU_NB; ++kk) x[kk] = (kk < nb) ? colj[kk] : 0.0;
#pragma unroll
  for (int kk = BLU_NB - 1; kk >= 0; --kk) {
    if (kk < nb) {
      x[kk] *= dinv[kk];
#pragma unroll
      for (int t = 0; t < kk; ++t) x[t] = fma(-U[t][kk], x[kk], x[t]);
    }
  }
#pragma unroll
  for (int kk = 0; kk < BLU_NB; ++kk)
    if (kk < nb) colj[kk] = x[kk];
}

// ---------------------------------------------------------------------------
// LU with partial pivoting and back substitution of a matrix below 64 rows, one wave per matrix
// ---------------------------------------------------------------------------
// Lane t holds row t of [A | R] in registers.  A step takes the pivot by a reduction over the lanes and the
// pivot row by lane reads; rows are not moved, each lane knows the position its row has come to.  The row moves
// down by one entry per step, so the loop over steps needs no register index, and the entries of U that leave it
// wait in LDS, each for its own lane: no barrier.  Blocks of CH columns that the step has left behind are
// skipped.  More right-hand sides than NC - n take several waves, each with its own factorisation.  Bound by
// the FP64 FMAs and lane reads of a step.  n = 25, 46 columns, the elements of 24 2D meshes: 0.82 ms (a
// 256-thread workgroup per matrix with eleven barriers per column: 1.68 ms).
template <int NC>
__global__ __launch_bounds__(64) void k_lu_small(double* Aall, int n, int ncols, long stride, int* info) {
  constexpr int CH = 8;
  extern __shared__ double U[];  // column k of U: U[64 k + lane]
  double* A = Aall + stride * blockIdx.x;
  const int lane = threadIdx.x;
  const int j0 = n + (NC - n) * static_cast<int>(blockIdx.y);  // the wave's right-hand sides
  const int R = min(NC - n, ncols - j0), w = n + R;
  double x[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j)
    x[j] = lane < n && j < w ? A[lane + static_cast<long>(n) * (j < n ? j : j0 + j - n)] : 0.0;
  int pos = lane < n ? lane : -1;
  int singular = 0;
  for (int k = 0; k < n; ++k) {
    // (a column without a comparable entry, all NaN, keeps its row)
    double bv = -1.0;
    int bp = k;
    const double v = fabs(x[0]);
    if (pos >= k && v > bv) {
      bv = v;
      bp = pos;
    }
    const int p = argmax_lanes(bv, bp);
    const int l = __builtin_ctzll(__ballot(pos == p));
    const double pv = lane_value(x[0], l);
    if (pv == 0.0) singular = 1;
    U[64 * k + lane] = x[0];
    pos = pos == p ? k : pos == k ? p : pos;
    const double f = pos > k ? x[0] / pv : 0.0;
#pragma unroll
    for (int c = 0; c < NC; c += CH)
      if (c + 1 < w - k) {
#pragma unroll
        for (int j = c; j < c + CH; ++j)
          if (j + 1 < NC) x[j] = fma(-f, lane_value(x[j + 1], l), x[j + 1]);
      }
  }
  for (int k = n - 1; k >= 0; --k) {
    const int l = __builtin_ctzll(__ballot(pos == k));
    const double u = U[64 * k + lane];
    double ukk = lane_value(u, l);
    if (fabs(ukk) < 0x1p-1021) {  // its reciprocal may overflow: the row times 2^128, which is exact
      ukk *= 0x1p128;
#pragma unroll
      for (int j = 0; j < NC; ++j) x[j] = pos == k ? x[j] * 0x1p128 : x[j];
    }
    const double inv = 1.0 / ukk;
    const double f = pos < k ? u : 0.0;
#pragma unroll
    for (int c = 0; c < NC; c += CH)
      if (c < R) {
#pragma unroll
        for (int j = c; j < c + CH; ++j) {
          const double y = lane_value(x[j], l);
          const double q = y * inv;
          const double t = fma(fma(-q, ukk, y), inv, q);  // y / ukk, the quotient corrected by its remainder
          x[j] = pos == k ? t : fma(-f, t, x[j]);
        }
      }
  }
  if (lane < n)
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (j < R) A[pos + static_cast<long>(n) * (j0 + j)] = x[j];
  if (lane == 0 && blockIdx.y == 0 && info) info[blockIdx.x] = singular;
}

template <int NC>
void lu_small(double* A, int n, int ncols, long stride, int batch, int* info, hipStream_t s) {
  const int chunks = (ncols - n + NC - n - 1) / (NC - n);
  k_lu_small<NC><<<dim3(batch, chunks), 64, static_cast<size_t>(n) * 64 * sizeof(double), s>>>(A, n, ncols, stride, info);
}

// RuS = D'^{-1} Ru from the stored FP32 LU factors of D' (replaying the blocked factorisation: each panel's
// row exchanges, then the unit-lower elimination), then the upper-triangular solve.  One wave per element:
// lane t holds entries t, t + 64, .. of the vector in registers, entry k reaches the others by a lane
// read, and 8 columns of the factors are loaded ahead, so a column costs no barrier (n = 100, 4096
// elements: 85 us, and 32 us for Rh -= K RuS, against 309 us together with a workgroup and two barriers per column;
// n = 250, with the product of 100 rows: 443 us).  The diagonal and its reciprocal wait in LDS.
// The panel width nbp (a multiple of 16) is the one lu_solve used for the factorisation.
template <int RPL>
__global__ __launch_bounds__(64) void k_refine_solve(int n, int nbp, const float* LU, const int* piv,
                                                     const double* Ru, double* RuS) {
  const long e = blockIdx.x;
  const int lane = threadIdx.x;
  const float* Le = LU + e * static_cast<long>(n) * n;
  __shared__ double diag[64 * RPL], dinv[64 * RPL];
  double y[RPL];
  int pv[RPL];
  int row[RPL];
#pragma unroll
  for (int q = 0; q < RPL; ++q) {
    const int r = lane + 64 * q;
    row[q] = min(r, n - 1);
    y[q] = Ru[e * n + row[q]];
    pv[q] = piv[e * n + row[q]];
    const double dq = static_cast<double>(Le[row[q] + static_cast<long>(n) * row[q]]);
    diag[r] = dq;
    dinv[r] = 1.0 / dq;
  }
  // entry k (uniform) of a vector held like y (every register's lane read, then the choice: choosing the
  // register first, the compiler may put the vector in memory and index it)
  auto pick = [&](const double (&v)[RPL], int k) {
    double x = lane_value(v[0], k & 63);
#pragma unroll
    for (int q = 1; q < RPL; ++q) {
      const double t = lane_value(v[q], k & 63);
      x = k >= 64 * q ? t : x;
    }
    return x;
  };
  float col[2][8][RPL];
  auto load = [&](int b, int k) {  // columns k .. k + 7 (past either end: the nearest one, unused)
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int q = 0; q < RPL; ++q)
        col[b][u][q] = Le[row[q] + static_cast<long>(n) * min(max(k + u, 0), n - 1)];
  };
  auto lower = [&](int b, int k) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k + u < n) {
        const double yk = pick(y, k + u);
#pragma unroll
        for (int q = 0; q < RPL; ++q)
          if (lane + 64 * q > k + u) y[q] = fma(-static_cast<double>(col[b][u][q]), yk, y[q]);
      }
  };
  load(0, 0);
  for (int k0 = 0; k0 < n; k0 += nbp) {
    const int nb = min(nbp, n - k0);
    for (int kk = k0; kk < k0 + nb; ++kk) {
      int p = pv[0];
#pragma unroll
      for (int q = 1; q < RPL; ++q)
        if (kk >= 64 * q) p = pv[q];
      p = k0 + __builtin_amdgcn_readlane(p, kk & 63);
      if (p != kk) {
        const double a = pick(y, kk), b = pick(y, p);
#pragma unroll
        for (int q = 0; q < RPL; ++q) y[q] = lane + 64 * q == kk ? b : lane + 64 * q == p ? a : y[q];
      }
    }
    for (int k = k0; k < k0 + nb; k += 16) {
      load(1, k + 8);
      lower(0, k);
      load(0, k + 16);
      if (k + 8 < k0 + nb) lower(1, k + 8);
    }
  }
  auto upper = [&](int b, int k) {  // columns k + 7 .. k
#pragma unroll
    for (int u = 7; u >= 0; --u)
      if (k + u >= 0) {
        const double dk = diag[k + u], di = dinv[k + u], yr = pick(y, k + u), qt = yr * di;
        const double yk = fma(fma(-qt, dk, yr), di, qt);  // yr / dk, the quotient corrected by its remainder
#pragma unroll
        for (int q = 0; q < RPL; ++q) {
          const int r = lane + 64 * q;
          if (r < k + u) y[q] = fma(-static_cast<double>(col[b][u][q]), yk, y[q]);
          else if (r == k + u) y[q] = yk;
        }
      }
  };
  __syncthreads();
  load(0, n - 8);
  for (int k = n - 8; k > -8; k -= 16) {
    load(1, k - 8);
    upper(0, k);
    load(0, k - 16);
    if (k - 8 > -8) upper(1, k - 8);
  }
#pragma unroll
  for (int q = 0; q < RPL; ++q)
    if (lane + 64 * q < n) RuS[e * n + lane + 64 * q] = y[q];
}

// The same for more than 256 unknowns: one workgroup per element, the vector in LDS
__global__ __launch_bounds__(256) void k_refine_solve_any(int n, int nbp, const float* LU, const int* piv,
                                                          const double* Ru, double* RuS) {
  const long e = blockIdx.x;
  extern __shared__ double sm[];
  double* y = sm;   // n
  const float* Le = LU + e * static_cast<long>(n) * n;
  const int* pe = piv + e * static_cast<long>(n);
  for (int t = threadIdx.x; t < n; t += 256) y[t] = Ru[e * n + t];
  __syncthreads();
  for (int k0 = 0; k0 < n; k0 += nbp) {
    const int nb = min(nbp, n - k0);
    if (threadIdx.x == 0)
      for (int kk = 0; kk < nb; ++kk) {
        const int p = k0 + pe[k0 + kk];
        if (p != k0 + kk) {
          const double t = y[k0 + kk];
          y[k0 + kk] = y[p];
          y[p] = t;
        }
      }
    __syncthreads();
    for (int k = k0; k < k0 + nb; ++k) {
      const double yk = y[k];
      for (int r = k + 1 + threadIdx.x; r < n; r += 256)
        y[r] = fma(-static_cast<double>(Le[r + static_cast<long>(n) * k]), yk, y[r]);
      __syncthreads();
    }
  }
  for (int k = n - 1; k >= 0; --k) {
    if (threadIdx.x == 0) y[k] /= static_cast<double>(Le[k + static_cast<long>(n) * k]);
    __syncthreads();
    const double yk = y[k];
    for (int r = threadIdx.x; r < k; r += 256)
      y[r] = fma(-static_cast<double>(Le[r + static_cast<long>(n) * k]), yk, y[r]);
    __syncthreads();
  }
  for (int t = threadIdx.x; t < n; t += 256) RuS[e * n + t] = y[t];
}

// panel width lu_solve uses for an n x n factorisation (see lu_solve).  64-wide panels (up to
// 150 KB of LDS at n = 300) were measured slower: one workgroup per CU leaves the latency-bound
// panel factorisation without company (C2 LU 0.36 s -> 0.55 s per assembly).
int lu_panel_width(int n) { return (static_cast<size_t>(n) * 32 * sizeof(double) <= 64000) ? 32 : 16; }
// the FP32 LU (the mixed form): 64-wide panels up to n = 250 (an n x 64 FP32 panel in 64 KB of LDS,
// 64 registers per row in the register panel), which halves the passes of the bandwidth-bound
// trailing update; 32 or 16 beyond
int lu_panel_width_f32(int n) {
  if (n <= 250) return 64;
  return (static_cast<size_t>(n) * 32 * sizeof(float) <= 64000) ? 32 : 16;
}

// a matrix's ints of piv_ws: the moved rows of a panel, their number and (new, old) of each.  An exchange moves
// two rows, so a panel of NB columns moves at most 2 NB of the n.
int piv_ints(int n, int NB) { return 1 + 2 * std::min(2 * NB, n); }

// operands of a GEMM inside the LU: FP64 storage and products, or FP32 storage and products
inline void lu_gemm_ptrs(Gemm& g, const double* A, const double* B, double* C) {
  g.A = A;
  g.B = B;
  g.C = C;
}
inline void lu_gemm_ptrs(Gemm& g, const float* A, const float* B, float* C) {
  g.Af = A;
  g.Bf = B;
  g.Cf = C;
  g.fp32 = 1;
}

template <typename T, int NB>
void blocked_lu(T* A, int n, int ncols, long stride, int batch, int* info, int* pivout, hipStream_t s,
                int* piv_ws, T* tri_ws) {
  // X[r0 : r0+nb, cols] = Tinv X[r0 : r0+nb, cols] in place (Tinv in tri_ws, ld NB)
  auto apply_tri = [&](int nb, int r0, long c0, int ncol) {
    Gemm g{};
    g.M = nb; g.N = ncol; g.K = nb; g.alpha = 1.0; g.beta = 0.0;
    T* X = A + r0 + static_cast<long>(n) * c0;
    lu_gemm_ptrs(g, tri_ws, X, X);
    g.lda = NB; g.sA0 = static_cast<long>(NB) * NB;
    g.ldb = n; g.sB0 = stride;
    g.ldc = n; g.sC0 = stride;
    g.nb0 = batch; g.nb1 = 1; g.nb2 = 1;
    gemm(g, s);
  };
  const int pws = piv_ints(n, NB);
  for (int k0 = 0; k0 < n; k0 += NB) {
    const int nb = std::min(NB, n - k0);
    if (piv_ws && n - k0 <= 256) {
      const int rows = n - k0;
      if (rows <= 64) k_lu_panel_wave<T, NB, 1><<<batch, 64, 0, s>>>(A, n, stride, k0, info, pivout, piv_ws, pws);
      else if (rows <= 128) k_lu_panel_wave<T, NB, 2><<<batch, 64, 0, s>>>(A, n, stride, k0, info, pivout, piv_ws, pws);
      else if (rows <= 192) k_lu_panel_wave<T, NB, 3><<<batch, 64, 0, s>>>(A, n, stride, k0, info, pivout, piv_ws, pws);
      else k_lu_panel_wave<T, NB, 4><<<batch, 64, 0, s>>>(A, n, stride, k0, info, pivout, piv_ws, pws);
      const int right = ncols - k0 - nb;
      if (right > 0) {
        k_lu_swap<T, NB><<<dim3(batch, (right + 63) / 64), 256, 0, s>>>(A, n, ncols, stride, k0, piv_ws, pws);
        if (tri_ws) {
          k_lu_tri_inv<T, NB, true><<<batch, 64, 0, s>>>(A, n, stride, k0, tri_ws);
          apply_tri(nb, k0, k0 + nb, right);
        } else {
          k_lu_u12<T, NB><<<dim3(batch, (right + 255) / 256), 256, 0, s>>>(A, n, ncols, stride, k0);
        }
      }
    } else {
      size_t shm = static_cast<size_t>(n - k0) * nb * sizeof(T);
      k_lu_panel<T, NB><<<batch, 256, shm, s>>>(A, n, ncols, stride, k0, info, pivout);
    }
    EXA_HIP(hipGetLastError());
    if (k0 + nb < n) {  // A22 -= L21 * U12
      Gemm g{};
      g.M = n - k0 - nb; g.N = ncols - k0 - nb; g.K = nb; g.alpha = -1.0; g.beta = 1.0;
      lu_gemm_ptrs(g, A + (k0 + nb) + static_cast<long>(n) * k0, A + k0 + static_cast<long>(n) * (k0 + nb),
                   A + (k0 + nb) + static_cast<long>(n) * (k0 + nb));
      g.lda = n; g.sA0 = stride;
      g.ldb = n; g.sB0 = stride;
      g.ldc = n; g.sC0 = stride;
      g.nb0 = batch; g.nb1 = 1; g.nb2 = 1;
      gemm(g, s);
    }
  }
  const int last = ((n - 1) / NB) * NB;
  for (int k0 = last; k0 >= 0; k0 -= NB) {
    if (tri_ws) {
      k_lu_tri_inv<T, NB, false><<<batch, 64, 0, s>>>(A, n, stride, k0, tri_ws);
      EXA_HIP(hipGetLastError());
      apply_tri(std::min(NB, n - k0), k0, n, ncols - n);
    } else {
      dim3 grid(static_cast<unsigned>(batch), static_cast<unsigned>((ncols - n + 255) / 256));
      k_lu_back<T, NB><<<grid, 256, 0, s>>>(A, n, ncols, stride, k0);
      EXA_HIP(hipGetLastError());
    }
    if (k0 > 0) {  // X[0:k0] -= U[0:k0, k0:k0+nb] * X[k0:k0+nb]
      const int nb = std::min(NB, n - k0);
      Gemm g{};
      g.M = k0; g.N = ncols - n; g.K = nb; g.alpha = -1.0; g.beta = 1.0;
      lu_gemm_ptrs(g, A + static_cast<long>(n) * k0, A + k0 + static_cast<long>(n) * n, A + static_cast<long>(n) * n);
      g.lda = n; g.sA0 = stride;
      g.ldb = n; g.sB0 = stride;
      g.ldc = n; g.sC0 = stride;
      g.nb0 = batch; g.nb1 = 1; g.nb2 = 1;
      gemm(g, s);
    }
  }
}

template <typename T>
void lu_blocked_any(T* A, int n, int ncols, long stride, int batch, int* info, hipStream_t s, int* pivout,
                    int* piv_ws, T* tri_ws) {
  // 32-wide panels when an n x 32 panel fits the 64 KB of LDS, else 16-wide; with a pivot
  // workspace, panels of up to 256 rows are factored in registers (64-wide register panels
  // were measured: no gain at n = 250, slower at n = 100)
  const int w = sizeof(T) == 4 ? lu_panel_width_f32(n) : lu_panel_width(n);
  if constexpr (sizeof(T) == 4) {
    if (w == 64) {
      blocked_lu<T, 64>(A, n, ncols, stride, batch, info, pivout, s, piv_ws, tri_ws);
      return;
    }
  }
  if (w == 32)
    blocked_lu<T, 32>(A, n, ncols, stride, batch, info, pivout, s, piv_ws, tri_ws);
  else if (static_cast<size_t>(n) * 16 * sizeof(T) <= 64000)
    blocked_lu<T, 16>(A, n, ncols, stride, batch, info, pivout, s, piv_ws, tri_ws);
  else
    throw Error(5, "dense block larger than 500 rows");
}

}  // namespace

int lu_piv_ws(int n, bool fp32) {
  if (!fp32 && n < BLU_MIN_N) return 0;  // k_lu_small
  return piv_ints(n, fp32 ? lu_panel_width_f32(n) : lu_panel_width(n));
}

void lu_solve(double* A, int n, int ncols, long stride, int batch, int* info, hipStream_t s, int* pivout,
              int* piv_ws, void* tri_ws) {
  if (batch <= 0) return;
  // the FP64 form keeps the substitution kernels (k_lu_u12, k_lu_back): explicit triangle inverses
  // amplify rounding by the triangle's condition number, which the FP64 form is not allowed to lose
  (void)tri_ws;
  if (ncols <= n) throw Error(5, "LU needs right-hand-side columns");
  if (n >= BLU_MIN_N || pivout) {
    lu_blocked_any(A, n, ncols, stride, batch, info, s, pivout, piv_ws, static_cast<double*>(nullptr));
    return;
  }
  // the narrowest registers that hold a row; beyond 96 columns the right-hand sides are split
  if (ncols <= 16) lu_small<16>(A, n, ncols, stride, batch, info, s);
  else if (ncols <= 32) lu_small<32>(A, n, ncols, stride, batch, info, s);
  else if (ncols <= 48) lu_small<48>(A, n, ncols, stride, batch, info, s);
  else if (ncols <= 64) lu_small<64>(A, n, ncols, stride, batch, info, s);
  else lu_small<96>(A, n, ncols, stride, batch, info, s);
  EXA_HIP(hipGetLastError());
}

void lu_solve(float* A, int n, int ncols, long stride, int batch, int* info, hipStream_t s, int* pivout,
              int* piv_ws, void* tri_ws) {
  if (batch <= 0) return;
  if (ncols <= n) throw Error(5, "FP32 LU needs right-hand-side columns");
  lu_blocked_any(A, n, ncols, stride, batch, info, s, pivout, piv_ws, static_cast<float*>(tri_ws));
}

void refine_rhs(const Dims& d, const float* LU, const int* piv, const float* K, const double* Ru, double* RuS,
                double* Rh, hipStream_t s) {
  if (d.ne <= 0) return;
  const int n = d.n, nbp = lu_panel_width_f32(n);
  if (n <= 64) k_refine_solve<1><<<d.ne, 64, 0, s>>>(n, nbp, LU, piv, Ru, RuS);
  else if (n <= 128) k_refine_solve<2><<<d.ne, 64, 0, s>>>(n, nbp, LU, piv, Ru, RuS);
  else if (n <= 192) k_refine_solve<3><<<d.ne, 64, 0, s>>>(n, nbp, LU, piv, Ru, RuS);
  else if (n <= 256) k_refine_solve<4><<<d.ne, 64, 0, s>>>(n, nbp, LU, piv, Ru, RuS);
  else k_refine_solve_any<<<d.ne, 256, n * sizeof(double), s>>>(n, nbp, LU, piv, Ru, RuS);
  EXA_HIP(hipGetLastError());
  trace_rhs(d, d.ne, K, RuS, n, Rh, s);
}

}  // namespace exa
