// krylov.hip -- the vector work and the scalars of restarted GMRES (gmres.cpp:361-597) on the device,
// for one problem or for every instance of a batch (segments of the trace vector).
//
// An Arnoldi step costs few launches: CGS three (dots, their sums, the update with the norm's
// partial sums) and MGS one per basis vector (the update by one vector with the dot with the next),
// each summing the partials of the launch before by itself; one last launch forms the norm, scales the
// new basis vector and applies the Givens rotations.  Every sum has a fixed order set by the length of its
// segment, so an instance's sums do not depend on the batch it is in.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace exa {

// ---------------------------------------------------------------------------
// Krylov scalars: the Givens rotations, the convergence test and the back substitution of every
// instance run on the device, so the host never waits on a step; stat[..] receives the number of
// instances still iterating.
// ---------------------------------------------------------------------------
namespace {

constexpr int GM_BS = 1024;  // one block: 16 waves

// cpuApplyGivensRotation (backend/Common/cpuimpl.h:167-197) on the new Hessenberg column of one
// instance: the rotations k < i are applied in order with the running entry (the column's entry k
// after rotation k-1) kept in a register, so the chain waits on FMAs only, not on memory; the
// column comes from hcol (entry k at hc[k*ns]) and the rotated column goes to H.
__device__ void dev_givens(const double* __restrict__ hc, int ns, double* __restrict__ H, double* __restrict__ s,
                           double* __restrict__ cs, double* __restrict__ sn, int i) {
  double carry = hc[0];
  int k = 0;
  for (; k + 8 <= i; k += 8) {  // the chunk's loads are issued before its FMAs
    double h1[8], c[8], sg[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      h1[u] = hc[static_cast<long>(k + u + 1) * ns];
      c[u] = cs[k + u];
      sg[u] = sn[k + u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      H[k + u] = c[u] * carry + sg[u] * h1[u];
      carry = -sg[u] * carry + c[u] * h1[u];
    }
  }
  for (; k < i; ++k) {
    const double h1 = hc[static_cast<long>(k + 1) * ns];
    const double c = cs[k], sg = sn[k];
    H[k] = c * carry + sg * h1;
    carry = -sg * carry + c * h1;
  }
  const double a = carry, b = hc[static_cast<long>(i + 1) * ns];
  double ci, si;
  if (b == 0.0) {
    ci = 1.0;
    si = 0.0;
  } else if (fabs(b) > fabs(a)) {
    const double t = a / b;
    si = 1.0 / sqrt(1.0 + t * t);
    ci = t * si;
  } else {
    const double t = b / a;
    ci = 1.0 / sqrt(1.0 + t * t);
    si = t * ci;
  }
  cs[i] = ci;
  sn[i] = si;
  const double t = ci * s[i];
  s[i + 1] = -si * s[i];
  s[i] = t;
  H[i] = ci * a + si * b;
  H[i + 1] = 0.0;
}

// cpuBackSolve (cpuimpl.h:199-208) by one wave: y (stride ys) = R^{-1} s over rows 0..i, R the
// leading (i+1) x (i+1) block of Hm (column-major, ld).  Column-oriented: lane l keeps the right-
// hand sides of rows l, l + 64, ...; for k = i .. 0 the owner of row k divides, the value goes to
// every lane, and each lane updates its rows above k; the columns' entries are loaded 8 columns
// ahead.  Rows beyond 64 * GM_ROWS fall back to one lane.
constexpr int GM_ROWS = 4;  // i + 1 <= 256 on the wave path
__device__ void dev_back_solve_wave(double* __restrict__ y, int ys, const double* __restrict__ Hm,
                                    const double* __restrict__ s, int i, int ld) {
  const int lane = threadIdx.x & 63;
  if (i + 1 > 64 * GM_ROWS) {
    if (lane == 0) {
      for (int j = i; j >= 0; --j) y[static_cast<long>(j) * ys] = s[j];
      for (int j = i; j >= 0; --j) {
        const double yj = y[static_cast<long>(j) * ys] / Hm[j + static_cast<long>(ld) * j];
        y[static_cast<long>(j) * ys] = yj;
        for (int k = j - 1; k >= 0; --k) y[static_cast<long>(k) * ys] -= Hm[k + static_cast<long>(ld) * j] * yj;
      }
    }
    return;
  }
  double r[GM_ROWS];
#pragma unroll
  for (int q = 0; q < GM_ROWS; ++q) {
    const int row = lane + 64 * q;
    r[q] = row <= i ? s[row] : 0.0;
  }
  for (int k0 = i; k0 >= 0; k0 -= 8) {
    double col[8][GM_ROWS], dg[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = k0 - u;
      const int kk = k >= 0 ? k : 0;
      dg[u] = Hm[kk + static_cast<long>(ld) * kk];
#pragma unroll
      for (int q = 0; q < GM_ROWS; ++q) {
        const int row = lane + 64 * q;
        col[u][q] = row < kk ? Hm[row + static_cast<long>(ld) * kk] : 0.0;
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = k0 - u;
      if (k < 0) break;
      const int ql = k >> 6, owner = k & 63;
      double rk = 0.0;
#pragma unroll
      for (int q = 0; q < GM_ROWS; ++q)
        if (q == ql) rk = r[q];
      rk = __shfl(rk, owner);
      const double yk = rk / dg[u];
      if (lane == owner) y[static_cast<long>(k) * ys] = yk;
#pragma unroll
      for (int q = 0; q < GM_ROWS; ++q) r[q] -= col[u][q] * yk;
    }
  }
}

__device__ void block_count(int mine, int* stat) {
  __shared__ int cnt;
  if (threadIdx.x == 0) cnt = 0;
  __syncthreads();
  if (mine) atomicAdd(&cnt, mine);
  __syncthreads();
  if (threadIdx.x == 0) stat[0] = cnt;
}

// start of a solve: an instance iterates unless ||b|| is zero, non-finite, or (Newton's own
// solves) below the nonlinear tolerance (gmres.cpp:412-415)
__global__ __launch_bounds__(GM_BS) void k_gmres_begin(GmresDev g, const double* nb, double tol, double ntol,
                                                       int use_ntol) {
  if (threadIdx.x == 0) {
    g.tol[0] = tol;
    g.jcount[0] = 0;
    g.ticket[0] = 0;
    g.bcount[0] = 0;
  }
  int mine = 0;
  for (int sg = threadIdx.x; sg < g.ns; sg += GM_BS) {
    const double b = nb[sg];
    const bool a = isfinite(b) && !(b == 0.0 || (use_ntol && b < ntol));
    g.act[sg] = a ? 1.0 : 0.0;
    g.jc[sg] = 0.0;
    g.iters[sg] = 0;
    mine += a;
  }
  block_count(mine, g.stat);
}

// first cycle: nrmb = ||P r0|| (gmres.cpp:431-445), s = (nrmb, 0, ...), coef = 1/||r|| scale of v_0
__global__ __launch_bounds__(GM_BS) void k_gmres_start(GmresDev g, const double* nr, double* coef) {
  int mine = 0;
  const int n1 = g.n1;
  for (int sg = threadIdx.x; sg < g.ns; sg += GM_BS) {
    const double r = nr[sg];
    if (g.act[sg] != 0.0 && !isfinite(r)) g.act[sg] = 0.0;
    const bool a = g.act[sg] != 0.0;
    g.nrmb[sg] = r;
    double* sv = g.sv + static_cast<long>(sg) * (n1 + 1);
    sv[0] = a ? r : 0.0;
    for (int k = 1; k <= n1; ++k) sv[k] = 0.0;
    coef[sg] = a ? r : 0.0;
    mine += a;
  }
  block_count(mine, g.stat);
}

// Arnoldi step j (column i of the cycle) of one instance, by one wave: rotate the new column h (LDS,
// entries k <= i + 1) with the stored rotations in order and form the new one
// (cpuApplyGivensRotation, cpuimpl.h:167-197), write the rotated column to Hm, test
// |s_{i+1}| / nrmb < tol; a converged instance gets y = R^{-1} s (zero above row i), jc = 1 (x += V y at
// the end of the cycle), act = 0 and the reference's iteration count j; a non-finite rotation stops the
// instance.  A column too long for LDS (h null) is read from hcol.  Adds 1 to bcount[0] when the instance
// iterates on.
constexpr int GM_LDS_N1 = 128;  // columns up to this length are staged in LDS
struct ArnoldiLds {
  double h[GM_LDS_N1 + 1], c[GM_LDS_N1], s[GM_LDS_N1];
  int flag;
};
__device__ void dev_arnoldi_wave(const GmresDev& g, int sg, int i, int j, double tol, const double* hcol,
                                 ArnoldiLds& lds) {
  const int n1 = g.n1, ns = g.ns;
  const int lane = threadIdx.x & 63;
  const bool staged = n1 <= GM_LDS_N1;
  double* H = g.Hm + static_cast<long>(sg) * n1 * n1 + static_cast<long>(n1) * i;
  double* sv = g.sv + static_cast<long>(sg) * (n1 + 1);
  double* cs = g.cs + static_cast<long>(sg) * (n1 + 1);
  double* sn = g.sn + static_cast<long>(sg) * (n1 + 1);
  if (staged)
    for (int k = lane; k < i; k += 64) {
      lds.c[k] = cs[k];
      lds.s[k] = sn[k];
    }
  __threadfence_block();
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) {
    if (staged) {
      double carry = lds.h[0];
      for (int k = 0; k < i; ++k) {
        const double h1 = lds.h[k + 1];
        lds.h[k] = lds.c[k] * carry + lds.s[k] * h1;
        carry = -lds.s[k] * carry + lds.c[k] * h1;
      }
      const double a0 = carry, b0 = lds.h[i + 1];
      double ci, si;
      if (b0 == 0.0) {
        ci = 1.0;
        si = 0.0;
      } else if (fabs(b0) > fabs(a0)) {
        const double t = a0 / b0;
        si = 1.0 / sqrt(1.0 + t * t);
        ci = t * si;
      } else {
        const double t = b0 / a0;
        ci = 1.0 / sqrt(1.0 + t * t);
        si = t * ci;
      }
      cs[i] = ci;
      sn[i] = si;
      const double t = ci * sv[i];
      sv[i + 1] = -si * sv[i];
      sv[i] = t;
      lds.h[i] = ci * a0 + si * b0;
      lds.h[i + 1] = 0.0;
    } else {
      dev_givens(hcol + sg, ns, H, sv, cs, sn, i);
    }
    g.iters[sg] = j + 1;
    const double s1 = sv[i + 1];
    int f = 1;  // 1 iterating, 2 converged, 0 stopped
    if (!isfinite(s1)) f = 0;
    else if (fabs(s1) / g.nrmb[sg] < tol) f = 2;
    if (f != 1) {
      g.act[sg] = 0.0;
      if (f == 2) {
        g.iters[sg] = j;
        g.jc[sg] = 1.0;
      }
    } else {
      atomicAdd(g.bcount, 1);
    }
    lds.flag = f;
  }
  __threadfence_block();
  __builtin_amdgcn_wave_barrier();
  if (staged)
    for (int k = lane; k <= i + 1; k += 64) H[k] = lds.h[k];
  if (lds.flag == 2) {  // y = R^{-1} s, zero above row i
    __threadfence_block();
    dev_back_solve_wave(g.y + sg, ns, g.Hm + static_cast<long>(sg) * n1 * n1, sv, i, n1);
    for (int k = i + 1 + lane; k < n1; k += 64) g.y[static_cast<long>(k) * ns + sg] = 0.0;
  }
}

// By one thread of each instance's block, after its dev_arnoldi_wave: the last one to come writes the
// count of iterating instances to stat[j % ring] and advances jcount.
__device__ void dev_arnoldi_count(const GmresDev& g, int j) {
  __threadfence();
  if (atomicAdd(g.ticket, 1) == g.ns - 1) {
    __threadfence();
    g.stat[j % g.ring] = atomicExch(g.bcount, 0);
    g.jcount[0] = j + 1;
    g.ticket[0] = 0;
  }
}

// end of a cycle of i steps: y = R^{-1} s over rows 0..i-1 for the instances still iterating
// (for x += V y, gmres.cpp:552, UpdateSolution); xmask marks them and the instances that converged
// in this cycle (their y is set), one wave per instance
__global__ __launch_bounds__(GM_BS) void k_gmres_cycle_y(GmresDev g, int i) {
  const int n1 = g.n1, ns = g.ns;
  const int lane = threadIdx.x & 63;
  for (int sg = static_cast<int>(threadIdx.x >> 6); sg < ns; sg += GM_BS / 64) {
    if (g.act[sg] != 0.0) {
      dev_back_solve_wave(g.y + sg, ns, g.Hm + static_cast<long>(sg) * n1 * n1,
                          g.sv + static_cast<long>(sg) * (n1 + 1), i - 1, n1);
      for (int k = i + lane; k < n1; k += 64) g.y[static_cast<long>(k) * ns + sg] = 0.0;
    }
    if (lane == 0) g.xmask[sg] = (g.act[sg] != 0.0 || g.jc[sg] != 0.0) ? 1.0 : 0.0;
  }
}

// end of a solve: x += V y still due for the instances that converged in the last cycle
__global__ __launch_bounds__(GM_BS) void k_gmres_flush(GmresDev g) {
  for (int sg = threadIdx.x; sg < g.ns; sg += GM_BS) {
    g.xmask[sg] = g.jc[sg];
    g.jc[sg] = 0.0;
  }
}

// restart test (gmres.cpp:561-566): ||P(b - A x)|| / nrmb < tol stops the instance; the others
// restart with s = (||r||, 0, ...) and v_0 = r / ||r||
__global__ __launch_bounds__(GM_BS) void k_gmres_restart(GmresDev g, const double* nr, double* coef) {
  int mine = 0;
  const int n1 = g.n1;
  const double tol = g.tol[0];
  const int j = g.jcount[0] - 1;  // the step this cycle ended with
  for (int sg = threadIdx.x; sg < g.ns; sg += GM_BS) {
    g.jc[sg] = 0.0;  // their x update was made with the cycle's
    const double r = nr[sg];
    if (g.act[sg] != 0.0 && r / g.nrmb[sg] < tol) g.act[sg] = 0.0;
    const bool a = g.act[sg] != 0.0;
    if (a) {
      double* sv = g.sv + static_cast<long>(sg) * (n1 + 1);
      sv[0] = r;
      for (int k = 1; k <= n1; ++k) sv[k] = 0.0;
    }
    coef[sg] = a ? r : 0.0;
    mine += a;
  }
  block_count(mine, g.stat + j % g.ring);
}

}  // namespace

void gmres_dev_begin(const GmresDev& g, const double* nb, double tol, double newton_tol, int use_newton_tol,
                     hipStream_t s) {
  k_gmres_begin<<<1, GM_BS, 0, s>>>(g, nb, tol, newton_tol, use_newton_tol);
  EXA_HIP(hipGetLastError());
}
void gmres_dev_start(const GmresDev& g, const double* nr, double* coef, hipStream_t s) {
  k_gmres_start<<<1, GM_BS, 0, s>>>(g, nr, coef);
  EXA_HIP(hipGetLastError());
}
void gmres_dev_cycle_y(const GmresDev& g, int i, hipStream_t s) {
  k_gmres_cycle_y<<<1, GM_BS, 0, s>>>(g, i);
  EXA_HIP(hipGetLastError());
}
void gmres_dev_flush(const GmresDev& g, hipStream_t s) {
  k_gmres_flush<<<1, GM_BS, 0, s>>>(g);
  EXA_HIP(hipGetLastError());
}
void gmres_dev_restart(const GmresDev& g, const double* nr, double* coef, hipStream_t s) {
  k_gmres_restart<<<1, GM_BS, 0, s>>>(g, nr, coef);
  EXA_HIP(hipGetLastError());
}
// ---------------------------------------------------------------------------
// Vectors split into per-instance segments.  Every block covers entries [bbeg, bend) of one segment (at
// most SEG_CHUNK), so a segment's sums and updates depend on its own entries and length only.
// ---------------------------------------------------------------------------
namespace {

constexpr int SEG_BS = 256;
constexpr int PIECES = static_cast<int>(SEG_CHUNK / 64);  // 64-entry pieces of a chunk
constexpr int GROUP = 2048;  // partials of a norm that one block sums
static_assert(SEG_CHUNK == 2 * SEG_BS, "two entries of a chunk per thread");

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// lane l's value (l uniform), to every lane
__device__ __forceinline__ double lane_value(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// sum of the block's 256 values v in a fixed order, to every thread (sh: 4 values of LDS, free again at
// the next barrier)
__device__ __forceinline__ double block_sum(double v, double* sh) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  return ((sh[0] + sh[1]) + sh[2]) + sh[3];
}

// sum of count partials by a block of 256 threads; the same order wherever it is done.  Eight loads are in
// flight per thread: one block on a norm's 19,700 partials of 1.3 million entries took 13.4 us per reduction on
// average over a step's two with one load at a time, 6.0 us here (and a block per GROUP 4.7 us, with 79,200).
__device__ __forceinline__ double partials_sum(const double* p, int count, double* sh) {
  double acc = 0.0;
  int i = threadIdx.x;
  for (; i + 7 * SEG_BS < count; i += 8 * SEG_BS) {
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = p[i + q * SEG_BS];
#pragma unroll
    for (int q = 0; q < 8; ++q) acc += v[q];
  }
  for (; i < count; i += SEG_BS) acc += p[i];
  return block_sum(acc, sh);
}

// partial[v*nblk + b] = <V_v, w> over block b for the vectors v < k.  Bound by reading V.  The chunk of w is
// staged in LDS; each wave sums C vectors at a time (four, or fewer vectors' share of them), with up to 16
// loads in flight per lane; the vectors are split over gridDim.y where the chunks alone leave the device idle.
// 24 instances, 330,000 entries together, 25 vectors on average: 16 us (one vector per wave at a time, one block
// per chunk: 40 us).
template <int C>
__global__ __launch_bounds__(SEG_BS) void k_seg_dots(SegMap m, const double* V, long ldv, int k, const double* w,
                                                     double* partial) {
  __shared__ double wl[SEG_CHUNK];
  const int b = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (m.act && m.act[m.bseg[b]] == 0.0) {  // block-uniform
    for (int v = threadIdx.x + SEG_BS * blockIdx.y; v < k; v += SEG_BS * gridDim.y)
      partial[static_cast<long>(v) * m.nblk + b] = 0.0;
    return;
  }
  const long i0 = m.bbeg[b];
  const int len = static_cast<int>(m.bend[b] - i0);
  for (int t = threadIdx.x; t < len; t += SEG_BS) wl[t] = w[i0 + t];
  __syncthreads();
  constexpr int U = C <= 2 ? 8 : 4;
  for (int v0 = 4 * C * blockIdx.y + C * wave; v0 < k; v0 += 4 * C * gridDim.y) {
    const double* x[C];
    double acc[C];
#pragma unroll
    for (int q = 0; q < C; ++q) {
      x[q] = V + ldv * min(v0 + q, k - 1) + i0;
      acc[q] = 0.0;
    }
    int t = lane;
    for (; t + 64 * (U - 1) < len; t += 64 * U) {
      double h[U][C];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < C; ++q) h[u][q] = x[q][t + 64 * u];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < C; ++q) acc[q] = fma(h[u][q], wl[t + 64 * u], acc[q]);
    }
    for (; t < len; t += 64)
#pragma unroll
      for (int q = 0; q < C; ++q) acc[q] = fma(x[q][t], wl[t], acc[q]);
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const double s = wave_sum(acc[q]);
      if (lane == 0 && v0 + q < k) partial[static_cast<long>(v0 + q) * m.nblk + b] = s;
    }
  }
}

// the same for fewer vectors than a wave takes at a time: one vector per blockIdx.y, two entries per thread
__global__ __launch_bounds__(SEG_BS) void k_seg_dot(SegMap m, const double* V, long ldv, const double* w,
                                                    double* partial) {
  __shared__ double sh[4];
  const int b = blockIdx.x;
  const double* x = V + ldv * blockIdx.y;
  double acc = 0.0;
  if (!m.act || m.act[m.bseg[b]] != 0.0) {
    const long i = m.bbeg[b] + threadIdx.x, end = m.bend[b];
    if (i < end) acc = x[i] * w[i];
    if (i + SEG_BS < end) acc = fma(x[i + SEG_BS], w[i + SEG_BS], acc);
  }
  acc = block_sum(acc, sh);
  if (threadIdx.x == 0) partial[static_cast<long>(blockIdx.y) * m.nblk + b] = acc;
}

// out[v*nseg + s] = sum of segment s's partials, sqrt if asked; the segment's partials are per per block
// and contiguous  (blockIdx.y = v)
__global__ __launch_bounds__(SEG_BS) void k_seg_reduce(SegMap m, const double* partial, int per, double* out,
                                                       int sqrt_out) {
  __shared__ double sh[4];
  const int sg = blockIdx.x;
  const double* pv = partial + static_cast<long>(blockIdx.y) * m.nblk * per;
  const double s = partials_sum(pv + static_cast<long>(per) * m.sbptr[sg], per * (m.sbptr[sg + 1] - m.sbptr[sg]), sh);
  if (threadIdx.x == 0) out[static_cast<long>(blockIdx.y) * m.nseg + sg] = sqrt_out ? sqrt(s) : s;
}

// x += alpha * sum_j V_j * y[j*nseg + seg]; NORM: npart[b*PIECES + piece] = <x, x> over the piece.  Bound by
// reading V.  One block per 64 entries, its four waves a quarter of the columns each with 8 loads in
// flight: 45,000 entries, 50 columns on average 6.5 us (a thread per entry walking all columns, with one
// load in flight and few blocks: 14.2 us).
// A turn's coefficients come with one load, a lane each, and lane reads: eight loads of all lanes through the
// caches that V streams through cost 445 us instead of 368 at 5,068,800 entries and 49 columns.
// KC > 0: at most KC columns in a quarter, and one wave takes all of them, four pieces to a block; the same sums.
// SKIPZ: columns whose coefficient is zero are not read (a basis column the solve has not written in this
// cycle may hold anything), and the waves take 8 columns in turn, which does not depend on k: a batch's longest
// solve sets k there, and an instance's sum may not depend on it.
template <bool SKIPZ, bool NORM, int KC>
__global__ __launch_bounds__(SEG_BS) void k_seg_gemv(SegMap m, double* __restrict__ x, const double* __restrict__ V,
                                                     long ldv, int k, const double* __restrict__ y, double alpha,
                                                     double* __restrict__ npart) {
  constexpr bool WHOLE = KC > 0;
  constexpr int PB = WHOLE ? 4 : 1;  // pieces of the block
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x / (PIECES / PB), piece = blockIdx.x % (PIECES / PB) * PB + (WHOLE ? wave : 0);
  const int sg = m.bseg[b];
  const long i0 = m.bbeg[b] + 64 * piece, end = m.bend[b];
  if (i0 >= end || (m.act && m.act[sg] == 0.0)) {  // uniform over the waves of a piece
    if (NORM && lane == 0 && (WHOLE || wave == 0)) npart[static_cast<long>(b) * PIECES + piece] = 0.0;
    return;
  }
  const double* Vi = V + min(i0 + lane, end - 1);
  const int kc = (k + 3) / 4;
  double s = 0.0;
  if constexpr (WHOLE) {
    const double yv = y[static_cast<long>(min(lane, k - 1)) * m.nseg + sg];
    double v[4][KC];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int u = 0; u < KC; ++u) v[q][u] = Vi[ldv * min(kc * q + u, k - 1)];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      double acc = 0.0;
#pragma unroll
      for (int u = 0; u < KC; ++u)
        acc = fma(v[q][u], u < kc && kc * q + u < k ? lane_value(yv, min(kc * q + u, 63)) : 0.0, acc);
      s += acc;
    }
  } else {
    __shared__ double red[4][64];
    const int j0 = SKIPZ ? 8 * wave : wave * kc, j1 = SKIPZ ? k : min(k, j0 + kc);
    double acc = 0.0;
    for (int j = j0; j < j1; j += SKIPZ ? 32 : 8) {
      const double yv = y[static_cast<long>(min(j + (lane & 7), j1 - 1)) * m.nseg + sg];
      double v[8], c[8];
      if (SKIPZ) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          c[u] = j + u < j1 ? lane_value(yv, u) : 0.0;
          v[u] = 0.0;
          if (c[u] != 0.0) v[u] = Vi[ldv * (j + u)];
        }
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = j + u < j1 ? Vi[ldv * (j + u)] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = j + u < j1 ? lane_value(yv, u) : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) acc = fma(v[u], c[u], acc);
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
    s = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
  }
  const bool in = i0 + lane < end;
  const double xn = in ? fma(alpha, s, x[i0 + lane]) : 0.0;
  if (in) x[i0 + lane] = xn;
  if (NORM) {
    const double q = wave_sum(xn * xn);
    if (lane == 0) npart[static_cast<long>(b) * PIECES + piece] = q;
  }
}

// Step k of modified Gram-Schmidt (getpoly.cpp:24-42): h_k = the sum of the partials pin (pre: already in
// hk[seg]), w -= h_k v_k, and the next step's partials pout = <w, vn> (vn null: <w, w>).
__global__ __launch_bounds__(SEG_BS) void k_seg_mgs(SegMap m, double* w, const double* vk, const double* vn,
                                                    const double* pin, double* pout, double* hk, int pre) {
  __shared__ double sh[4], sh2[4];
  const int b = blockIdx.x, sg = m.bseg[b];
  const int first = m.sbptr[sg];
  if (m.act && m.act[sg] == 0.0) {  // block-uniform
    if (threadIdx.x == 0) {
      pout[b] = 0.0;
      if (b == first) hk[sg] = 0.0;
    }
    return;
  }
  const long i = m.bbeg[b] + threadIdx.x, end = m.bend[b];
  double wv[2], v[2], n[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const bool in = i + SEG_BS * q < end;
    wv[q] = in ? w[i + SEG_BS * q] : 0.0;
    v[q] = in ? vk[i + SEG_BS * q] : 0.0;
    n[q] = in && vn ? vn[i + SEG_BS * q] : 0.0;
  }
  const double h = pre ? hk[sg] : partials_sum(pin + first, m.sbptr[sg + 1] - first, sh);
  if (!pre && b == first && threadIdx.x == 0) hk[sg] = h;
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const double x = fma(-h, v[q], wv[q]);
    if (i + SEG_BS * q < end) w[i + SEG_BS * q] = x;
    acc = fma(x, vn ? n[q] : x, acc);
  }
  acc = block_sum(acc, sh2);
  if (threadIdx.x == 0) pout[b] = acc;
}

// gsum[s*gmax + g] = the g-th GROUP of segment s's partials (per per block, contiguous), by block (s, g)
__global__ __launch_bounds__(SEG_BS) void k_seg_groups(SegMap m, const double* partial, int per, double* gsum, int gmax) {
  __shared__ double sh[4];
  const int sg = blockIdx.x, i0 = GROUP * blockIdx.y;
  const int count = per * (m.sbptr[sg + 1] - m.sbptr[sg]);
  if (i0 >= count) return;  // block-uniform
  const double s = partials_sum(partial + static_cast<long>(per) * m.sbptr[sg] + i0, min(GROUP, count - i0), sh);
  if (threadIdx.x == 0) gsum[static_cast<long>(sg) * gmax + blockIdx.y] = s;
}

// sum of a segment's count group sums, by every wave for itself: a few as uniform values (194,400 entries, two
// groups, 25 columns: a step 29.0 us as with one reduction in a launch of its own; by the block 29.3), many by the lanes
__device__ __forceinline__ double groups_sum(const double* p, int count) {
  double acc = 0.0;
  if (count <= 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = u < count ? p[u] : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
    return acc;
  }
  for (int i = threadIdx.x & 63; i < count; i += 64) acc += p[i];
  return wave_sum(acc);
}

// End of an Arnoldi step: the norm of w from its partials (per per block; LONG: from the sums of their
// groups, gmax of them per segment), w /= norm (0 where the norm is 0), and each instance's rotations and
// convergence test.  Blocks [0, nseg): one instance each; the others: a chunk of w each.
template <bool LONG>
__global__ __launch_bounds__(SEG_BS) void k_seg_finish(SegMap m, GmresDev g, int i, double* w, const double* npart,
                                                       int per, int gmax, double* hcol) {
  __shared__ double sh[4];
  __shared__ ArnoldiLds lds;
  const int blk = static_cast<int>(blockIdx.x) - m.nseg;
  const int sg = blk < 0 ? static_cast<int>(blockIdx.x) : m.bseg[blk];
  const int first = m.sbptr[sg], count = per * (m.sbptr[sg + 1] - first);
  double* hn = hcol + static_cast<long>(i + 1) * m.nseg + sg;
  double wv[2];
  if (LONG && blk >= 0)  // the chunk's values come while the norm is summed
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const long t = m.bbeg[blk] + threadIdx.x + SEG_BS * q;
      wv[q] = t < m.bend[blk] ? w[t] : 0.0;
    }
  const double nrm = sqrt(LONG ? groups_sum(npart + static_cast<long>(sg) * gmax, (count + GROUP - 1) / GROUP)
                               : partials_sum(npart + static_cast<long>(per) * first, count, sh));
  if (blk >= 0) {
    const double c = nrm != 0.0 ? 1.0 / nrm : 0.0;
    if (LONG) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const long t = m.bbeg[blk] + threadIdx.x + SEG_BS * q;
        if (t < m.bend[blk]) w[t] = wv[q] * c;
      }
    } else {
      for (long t = m.bbeg[blk] + threadIdx.x; t < m.bend[blk]; t += SEG_BS) w[t] *= c;
    }
    return;
  }
  const int j = g.jcount[0];
  const bool live = g.act[sg] != 0.0;
  if (live) {
    if (g.n1 <= GM_LDS_N1)
      for (int k = threadIdx.x; k <= i; k += SEG_BS) lds.h[k] = hcol[static_cast<long>(k) * m.nseg + sg];
    if (threadIdx.x == 0) {
      lds.h[min(i + 1, GM_LDS_N1)] = nrm;
      *hn = nrm;
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    if (live) dev_arnoldi_wave(g, sg, i, j, g.tol[0], hcol, lds);
    if (threadIdx.x == 0) dev_arnoldi_count(g, j);
  }
}

// A whole modified Gram-Schmidt step of one short vector (n <= 8 * 1024) in one workgroup: w stays in
// registers, the next basis vector is read ahead of the current dot's sum.  The step of 16 x 16 quads, p = 3
// (2176 entries, 4 basis vectors on average) takes 7.6 us; as a dot, a sum and an update per vector, a norm, a
// scaling and the rotations it was 17 launches and 35 us.
constexpr int ONE_BS = 1024, ONE_PER = 8;
__global__ __launch_bounds__(ONE_BS) void k_mgs_one(GmresDev g, const double* V, long n, int i, double* w) {
  __shared__ double sh[2][ONE_BS / 64];
  __shared__ ArnoldiLds lds;
  const int j = g.jcount[0];
  const bool live = g.act[0] != 0.0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (live) {
    double x[ONE_PER], v[ONE_PER];
#pragma unroll
    for (int q = 0; q < ONE_PER; ++q) {
      const long t = threadIdx.x + ONE_BS * q;
      x[q] = t < n ? w[t] : 0.0;
      v[q] = t < n ? V[t] : 0.0;
    }
    for (int k = 0; k <= i + 1; ++k) {  // step i + 1: the norm
      double acc = 0.0;
#pragma unroll
      for (int q = 0; q < ONE_PER; ++q) acc = fma(x[q], k <= i ? v[q] : x[q], acc);
      acc = wave_sum(acc);
      if (lane == 0) sh[k & 1][wave] = acc;
      double nx[ONE_PER];
      const double* Vn = V + n * min(k + 1, i);
#pragma unroll
      for (int q = 0; q < ONE_PER; ++q) {
        const long t = threadIdx.x + ONE_BS * q;
        nx[q] = t < n ? Vn[t] : 0.0;
      }
      __syncthreads();
      double h = 0.0;
#pragma unroll
      for (int q = 0; q < ONE_BS / 64; ++q) h += sh[k & 1][q];
      if (k > i) h = sqrt(h);
      if (threadIdx.x == 0) lds.h[k] = h;
      const double c = h != 0.0 ? 1.0 / h : 0.0;
#pragma unroll
      for (int q = 0; q < ONE_PER; ++q) {
        x[q] = k <= i ? fma(-h, v[q], x[q]) : x[q] * c;
        v[q] = nx[q];
      }
    }
#pragma unroll
    for (int q = 0; q < ONE_PER; ++q) {
      const long t = threadIdx.x + ONE_BS * q;
      if (t < n) w[t] = x[q];
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    if (live) dev_arnoldi_wave(g, 0, i, j, g.tol[0], nullptr, lds);
    if (threadIdx.x == 0) dev_arnoldi_count(g, j);
  }
}

// y += scale * coef[seg] * x
__global__ __launch_bounds__(SEG_BS) void k_seg_axpy(SegMap m, double* y, const double* x, const double* coef,
                                                     double scale) {
  const int b = blockIdx.x;
  if (m.act && m.act[m.bseg[b]] == 0.0) return;
  const double c = scale * coef[m.bseg[b]];
  if (c == 0.0) return;
  for (long i = m.bbeg[b] + threadIdx.x; i < m.bend[b]; i += SEG_BS) y[i] = fma(c, x[i], y[i]);
}

// mode 0: y = coef[seg] * x;  mode 1: y = x / coef[seg] (0 where coef[seg] == 0)
__global__ __launch_bounds__(SEG_BS) void k_seg_scale(SegMap m, double* y, const double* x, const double* coef,
                                                      int mode) {
  const int b = blockIdx.x;
  const double cv = coef[m.bseg[b]];
  const double c = mode == 0 ? cv : (cv != 0.0 ? 1.0 / cv : 0.0);
  for (long i = m.bbeg[b] + threadIdx.x; i < m.bend[b]; i += SEG_BS) y[i] = c * x[i];
}

// Partials of a segment up to this count (and one GROUP of a norm's) are summed again by every block that needs
// the sum (one more read of a few KB from the L2); longer segments' sums get a launch of their own, in which
// every GROUP of a norm's partials is a block's.  A segment's order is the same in both.
constexpr int MGS_AGAIN = 1024;

int norm_groups(const SegMap& m) { return (m.maxblk * PIECES + GROUP - 1) / GROUP; }

template <int C>
void launch_dots(const SegMap& m, const double* V, long ldv, int k, const double* w, double* partial, hipStream_t s) {
  // about 1024 blocks, one turn of the waves to a block at least
  const int ny = std::max(1, std::min((k + 4 * C - 1) / (4 * C), 1024 / m.nblk));
  k_seg_dots<C><<<dim3(m.nblk, ny), SEG_BS, 0, s>>>(m, V, ldv, k, w, partial);
}

// k_seg_gemv with one wave per piece: few columns leave most of a wave's loads in flight unused otherwise.  A
// step with 3, 5, 9 and 13 columns, four waves per piece / one: 24 instances, 330,000 entries 21.7/19.7,
// 22.0/20.6, 24.5/23.8, 27.8/27.8 us; one problem, 5 columns, 630,000 entries 32.6/29.6, 1,260,000 49.2/42.2,
// 5,068,800 141/112; 40,000 14.8/15.5.
constexpr int WHOLE_COLS = 12, WHOLE_CHUNKS = 640;

template <int KC>
void launch_gemv_whole(const SegMap& m, double* x, const double* V, long ldv, int k, const double* y, double* npart,
                       hipStream_t s) {
  k_seg_gemv<false, true, KC><<<m.nblk * (PIECES / 4), SEG_BS, 0, s>>>(m, x, V, ldv, k, y, -1.0, npart);
}
void launch_cgs_update(const SegMap& m, double* x, const double* V, long ldv, int k, const double* y, double* npart,
                       hipStream_t s) {
  if (k > WHOLE_COLS || m.nblk < WHOLE_CHUNKS)
    k_seg_gemv<false, true, 0><<<m.nblk * PIECES, SEG_BS, 0, s>>>(m, x, V, ldv, k, y, -1.0, npart);
  else if (k <= 4) launch_gemv_whole<1>(m, x, V, ldv, k, y, npart, s);
  else if (k <= 8) launch_gemv_whole<2>(m, x, V, ldv, k, y, npart, s);
  else launch_gemv_whole<3>(m, x, V, ldv, k, y, npart, s);
}

}  // namespace

long seg_partials(const SegMap& m, int k) {
  return static_cast<long>(std::max(m.nblk, 1)) * std::max(k, PIECES) + static_cast<long>(m.nseg) * norm_groups(m);
}

void seg_multidot(const SegMap& m, const double* V, long ldv, int k, const double* w, double* partial,
                  double* out, int sqrt_out, hipStream_t s) {
  if (m.nblk == 0 || k == 0) return;
  if (k < 4) k_seg_dot<<<dim3(m.nblk, k), SEG_BS, 0, s>>>(m, V, ldv, w, partial);
  else if (k == 4) launch_dots<1>(m, V, ldv, k, w, partial, s);
  else if (k <= 8) launch_dots<2>(m, V, ldv, k, w, partial, s);
  else if (k <= 12) launch_dots<3>(m, V, ldv, k, w, partial, s);
  else launch_dots<4>(m, V, ldv, k, w, partial, s);
  k_seg_reduce<<<dim3(m.nseg, k), SEG_BS, 0, s>>>(m, partial, 1, out, sqrt_out);
  EXA_HIP(hipGetLastError());
}

void seg_arnoldi(const SegMap& m, const GmresDev& g, const double* V, long n, int i, int mgs, double* w,
                 double* partial, double* hcol, hipStream_t s) {
  if (m.nblk == 0) return;
  const int ns = m.nseg;
  if (mgs && !m.shared && n <= ONE_BS * ONE_PER && g.n1 <= GM_LDS_N1) {
    k_mgs_one<<<1, ONE_BS, 0, s>>>(g, V, n, i, w);
    EXA_HIP(hipGetLastError());
    return;
  }
  int per = 1;
  double* np;
  if (mgs) {
    double *pin = partial, *pout = partial + m.nblk;
    k_seg_dot<<<m.nblk, SEG_BS, 0, s>>>(m, V, n, w, pin);
    const int pre = m.maxblk > MGS_AGAIN;
    for (int k = 0; k <= i; ++k) {
      double* hk = hcol + static_cast<long>(k) * ns;
      if (pre) k_seg_reduce<<<ns, SEG_BS, 0, s>>>(m, pin, 1, hk, 0);
      k_seg_mgs<<<m.nblk, SEG_BS, 0, s>>>(m, w, V + n * k, k < i ? V + n * (k + 1) : nullptr, pin, pout, hk, pre);
      std::swap(pin, pout);
    }
    np = pin;
  } else {
    seg_multidot(m, V, n, i + 1, w, partial, hcol, 0, s);
    np = partial;
    per = PIECES;
    launch_cgs_update(m, w, V, n, i + 1, hcol, np, s);
  }
  int gmax = 0;
  if (m.maxblk * per > GROUP) {
    gmax = (m.maxblk * per + GROUP - 1) / GROUP;
    double* gsum = partial + static_cast<long>(m.nblk) * std::max(i + 2, PIECES);
    k_seg_groups<<<dim3(ns, gmax), SEG_BS, 0, s>>>(m, np, per, gsum, gmax);
    np = gsum;
  }
  if (gmax) k_seg_finish<true><<<ns + m.nblk, SEG_BS, 0, s>>>(m, g, i, w, np, per, gmax, hcol);
  else k_seg_finish<false><<<ns + m.nblk, SEG_BS, 0, s>>>(m, g, i, w, np, per, 0, hcol);
  EXA_HIP(hipGetLastError());
}

void seg_axpy(const SegMap& m, double* y, const double* x, const double* coef, double scale, hipStream_t s) {
  if (m.nblk == 0) return;
  k_seg_axpy<<<m.nblk, SEG_BS, 0, s>>>(m, y, x, coef, scale);
  EXA_HIP(hipGetLastError());
}

void seg_scale(const SegMap& m, double* y, const double* x, const double* coef, int mode, hipStream_t s) {
  if (m.nblk == 0) return;
  k_seg_scale<<<m.nblk, SEG_BS, 0, s>>>(m, y, x, coef, mode);
  EXA_HIP(hipGetLastError());
}

void seg_gemv_cols(const SegMap& m, double* x, const double* V, long ldv, int k, const double* y, double alpha,
                   hipStream_t s) {
  if (m.nblk == 0 || k == 0) return;
  k_seg_gemv<true, false, 0><<<m.nblk * PIECES, SEG_BS, 0, s>>>(m, x, V, ldv, k, y, alpha, nullptr);
  EXA_HIP(hipGetLastError());
}

}  // namespace exa
