// matvec.hip -- the element products of the condensed operator and of the inverted Schwarz blocks
// (hdgMatVec's element part, backend/Discretization/matvec.cpp:377-380).
#include "blkval.hpp"
#include "common.hpp"
#include "kernels.hpp"

namespace exa {

namespace {

// Entry t of block e's input vector: trace unknown c = t % ncu of node con[..] (con null: of a face's own
// nodes), from the trace vector v, or summed from the element products of a preceding matvec (in.src1: the
// gather of face_gather, in its order, without the pass that writes the trace vector).
__device__ __forceinline__ double trace_in(const TraceIn& in, int t, long e, int m, int ncu, int ndf) {
  const int c = t % ncu, jl = t / ncu;
  const long g = in.con ? in.con[jl + static_cast<long>(ndf) * e] : jl + static_cast<long>(m / ncu) * e;
  if (!in.src1) return in.v[c + ncu * g];
  double x = in.v[in.src1[g] + c];
  const long s2 = in.src2[g];
  if (s2 >= 0) x += in.v[s2 + c];
  return x;
}

// hdgMatVec element part (matvec.cpp:377-380): we_e = H_e * v_e with v_e gathered
// through elemcon.  One workgroup per element; each of the 4 waves owns a
// quarter of the columns, lanes own VW consecutive rows (16-byte vector loads of
// the column), accumulation is FP64, and the four partial sums are added in LDS
// in a fixed order.
// NRB > 0: exactly NRB row blocks of 64 VW rows (m > 64 VW (NRB - 1)), with CB columns' loads
// issued before their FMAs (more bytes in flight per wave; a row's FMAs still run over the columns
// in order); NRB = 0: any m <= 1024, one column at a time.
template <typename T, int VW, int NRB>
__global__ __launch_bounds__(256) void k_matvec_elem(int m, int ncu, int ndf, const T* H, TraceIn in, double* we,
                                                     const int* einst, const double* emask, const double* act) {
  if (act && act[0] == 0.0) return;  // a finished solve (grid-uniform)
  typedef T vecT __attribute__((ext_vector_type(VW)));
  constexpr int MAXRB = NRB > 0 ? NRB : (1024 + 64 * VW - 1) / (64 * VW);  // m <= 1024
  constexpr int CB = NRB > 0 ? (sizeof(T) <= 4 ? 4 : 2) : 1;
  const long e = blockIdx.x;
  if (emask && einst && emask[einst[e]] == 0.0) {  // block-uniform: the element's instance is inactive
    for (int r = threadIdx.x; r < m; r += 256) we[e * m + r] = 0.0;
    return;
  }
  extern __shared__ double sm[];
  double* ve = sm;          // m
  double* red = sm + m;     // 4*m
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int t = tid; t < m; t += 256)
    ve[t] = trace_in(in, t, e, m, ncu, ndf);
  __syncthreads();
  const int cper = (m + 3) / 4;
  const int c0 = wave * cper, c1 = min(m, c0 + cper);
  const int nrb = (m + 64 * VW - 1) / (64 * VW);
  double acc[MAXRB][VW];
#pragma unroll
  for (int rb = 0; rb < MAXRB; ++rb)
#pragma unroll
    for (int q = 0; q < VW; ++q) acc[rb][q] = 0.0;
  const T* He = H + e * static_cast<long>(m) * m;
  int cfirst = c0;
  if (CB > 1) {
    for (; cfirst + CB <= c1; cfirst += CB) {
      vecT h[CB][MAXRB];
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const T* col = He + static_cast<long>(m) * (cfirst + j);
#pragma unroll
        for (int rb = 0; rb < MAXRB; ++rb) {
          const int r = VW * (lane + 64 * rb);
          if (r < m) h[j][rb] = *reinterpret_cast<const vecT*>(col + r);
        }
      }
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        const double vc = ve[cfirst + j];
#pragma unroll
        for (int rb = 0; rb < MAXRB; ++rb) {
          const int r = VW * (lane + 64 * rb);
          if (r < m)
#pragma unroll
            for (int q = 0; q < VW; ++q) acc[rb][q] = fma(blk_val(h[j][rb][q]), vc, acc[rb][q]);
        }
      }
    }
  }
  for (int c = cfirst; c < c1; ++c) {
    const double vc = ve[c];
    const T* col = He + static_cast<long>(m) * c;
#pragma unroll
    for (int rb = 0; rb < MAXRB; ++rb) {
      const int r = VW * (lane + 64 * rb);
      if (rb < nrb && r < m) {
        const vecT h = *reinterpret_cast<const vecT*>(col + r);
#pragma unroll
        for (int q = 0; q < VW; ++q) acc[rb][q] = fma(blk_val(h[q]), vc, acc[rb][q]);
      }
    }
  }
#pragma unroll
  for (int rb = 0; rb < MAXRB; ++rb) {
    const int r = VW * (lane + 64 * rb);
    if (rb < nrb && r < m)
#pragma unroll
      for (int q = 0; q < VW; ++q) red[wave * m + r + q] = acc[rb][q];
  }
  __syncthreads();
  for (int r = tid; r < m; r += 256)
    we[e * m + r] = ((red[r] + red[m + r]) + red[2 * m + r]) + red[3 * m + r];
}

// The same product for trace blocks whose column fits one wave's vector loads (m <= 64 VW: 2D
// elements and low-order 3D ones).  Bound by reading H.  WPE waves share an element and split its
// columns; within a wave, m / VW lanes hold the rows of a column and G = 64 VW / m columns are read
// side by side, so a wave's 16-byte loads cover G m consecutive entries, and U of these loads are in
// flight before the first FMA.  At m = 96, FP64, 2025 elements: 24 us = 6.2 TB/s (one thread per row,
// reading single entries with one load in flight, took 69 us); m = 192, BF16, 1864 elements: 23 us (the
// row-block kernel, with 24 of 64 lanes reading, 38 us).  Every sum's order is fixed
// by m and the storage alone, so an instance's products do not depend on the batch it is in.
// emask/einst (optional): elements of an instance whose mask is 0 only write zeros (instances that
// have left a batched GMRES).
template <typename T, int VW, int WPE>
__global__ __launch_bounds__(256) void k_matvec_small(int m, int ncu, int ndf, int ne, const T* H, TraceIn in,
                                                      double* we, const int* einst, const double* emask,
                                                      const double* act) {
  if (act && act[0] == 0.0) return;  // a finished solve (grid-uniform)
  typedef T vecT __attribute__((ext_vector_type(VW)));
  constexpr int EPB = 4 / WPE;  // elements of the workgroup
  constexpr int U = 8;
  extern __shared__ double sm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int sub = wave / WPE, part = wave % WPE;
  const int NL = m / VW, G = 64 / NL;
  const long e = blockIdx.x * static_cast<long>(EPB) + sub;
  const bool on = e < ne && !(emask && einst && emask[einst[e]] == 0.0);
  double* ve = sm + sub * (1 + WPE * G) * m;  // m
  double* red = ve + m;                       // WPE G m
  const int te = tid - sub * (64 * WPE);
  if (on)
    for (int t = te; t < m; t += 64 * WPE) ve[t] = trace_in(in, t, e, m, ncu, ndf);
  __syncthreads();
  const int rg = lane % NL, cg = lane / NL;
  if (on && cg < G) {
    const int cper = (m + WPE - 1) / WPE;
    const int c0 = part * cper, c1 = min(m, c0 + cper);
    const T* He = H + e * static_cast<long>(m) * m + VW * rg;
    double acc[VW];
#pragma unroll
    for (int q = 0; q < VW; ++q) acc[q] = 0.0;
    int cb = c0;
    for (; cb + U * G <= c1; cb += U * G) {
      vecT h[U];
#pragma unroll
      for (int j = 0; j < U; ++j)
        h[j] = *reinterpret_cast<const vecT*>(He + static_cast<long>(m) * (cb + cg + G * j));
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const double vc = ve[cb + cg + G * j];
#pragma unroll
        for (int q = 0; q < VW; ++q) acc[q] = fma(blk_val(h[j][q]), vc, acc[q]);
      }
    }
    if (cb < c1) {  // the last round: columns past the part's end reread its last one, unused
      vecT h[U];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const int c = min(cb + cg + G * j, c1 - 1);
        h[j] = *reinterpret_cast<const vecT*>(He + static_cast<long>(m) * c);
      }
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const int c = cb + cg + G * j;
        if (c < c1) {
          const double vc = ve[c];
#pragma unroll
          for (int q = 0; q < VW; ++q) acc[q] = fma(blk_val(h[j][q]), vc, acc[q]);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < VW; ++q) red[(part * G + cg) * m + VW * rg + q] = acc[q];
  }
  __syncthreads();
  if (e < ne)
    for (int t = te; t < m; t += 64 * WPE) {
      double s = 0.0;
      if (on)
        for (int g = 0; g < WPE * G; ++g) s += red[g * m + t];
      we[e * m + t] = s;
    }
}

struct Blocks {  // m x m blocks of ne elements (or faces)
  int m, ncu, ndf, ne;
  const int* einst;
  const double *emask, *act;
};

template <typename T, int VW, int NRB>
void launch_rows(const Blocks& b, const T* H, const TraceIn& in, double* we, hipStream_t s) {
  const size_t shm = static_cast<size_t>(5) * b.m * sizeof(double);
  k_matvec_elem<T, VW, NRB><<<b.ne, 256, shm, s>>>(b.m, b.ncu, b.ndf, H, in, we, b.einst, b.emask, b.act);
}

template <typename T, int VW, int WPE>
void launch_small(const Blocks& b, const T* H, const TraceIn& in, double* we, hipStream_t s) {
  constexpr int EPB = 4 / WPE;
  const int G = 64 / (b.m / VW);
  const size_t shm = static_cast<size_t>(EPB) * (1 + WPE * G) * b.m * sizeof(double);
  k_matvec_small<T, VW, WPE><<<(b.ne + EPB - 1) / EPB, 256, shm, s>>>(b.m, b.ncu, b.ndf, b.ne, H, in, we, b.einst,
                                                                       b.emask, b.act);
}

// A block of at most 8 KB keeps one wave per element (its few loads are one round anyway);
// larger blocks split their columns over four.
template <typename T, int VW>
void small_vw(const Blocks& b, const T* H, const TraceIn& in, double* we, hipStream_t s) {
  if (static_cast<size_t>(b.m) * b.m * sizeof(T) <= 8192) launch_small<T, VW, 1>(b, H, in, we, s);
  else launch_small<T, VW, 4>(b, H, in, we, s);
}

// the widest load (up to 16 bytes: 2 doubles, 4 floats, 8 BF16) that the rows of a column divide
// into: a column starts at a multiple of m, so the loads are aligned
template <typename T>
int rows_per_load(int m) {
  constexpr int VMAX = 16 / sizeof(T);
  return m % VMAX == 0 ? VMAX : (VMAX > 4 && m % 4 == 0) ? 4 : m % 2 == 0 ? 2 : 1;
}

template <typename T>
void products(const Blocks& b, const T* H, const TraceIn& in, double* we, hipStream_t s) {
  if (b.ne <= 0) return;
  if (b.m > 1024) throw Error(5, "element trace block larger than 1024");
  constexpr int VMAX = 16 / sizeof(T);
  const int vw = rows_per_load<T>(b.m);
  if (b.m <= 64 * vw) {  // a column is at most one load of a wave
    if (vw == VMAX) {
      small_vw<T, VMAX>(b, H, in, we, s);
    } else if (vw == 4) {
      if constexpr (VMAX > 4) small_vw<T, 4>(b, H, in, we, s);
    } else if (vw == 2) {
      if constexpr (VMAX > 2) small_vw<T, 2>(b, H, in, we, s);
    } else {
      small_vw<T, 1>(b, H, in, we, s);
    }
  } else if (vw == VMAX) {
    const int nrb = (b.m + 64 * VMAX - 1) / (64 * VMAX);
    if (nrb == 2) launch_rows<T, VMAX, 2>(b, H, in, we, s);
    else if (nrb == 3) launch_rows<T, VMAX, 3>(b, H, in, we, s);
    else launch_rows<T, VMAX, 0>(b, H, in, we, s);
  } else if (vw == 4) {  // BF16 blocks: 8-byte loads
    if constexpr (VMAX > 4) launch_rows<T, 4, 0>(b, H, in, we, s);
  } else if (vw == 2) {
    if constexpr (VMAX > 2) launch_rows<T, 2, 0>(b, H, in, we, s);
  } else {
    launch_rows<T, 1, 0>(b, H, in, we, s);
  }
  EXA_HIP(hipGetLastError());
}

// Rh_e -= K_e u_e (the condensation's trace residual; u_e the last column of the element's solved
// [D | F | Ru]).  One workgroup per element: its four waves split the n columns, lanes hold VW rows
// and, below 64 VW rows, G columns side by side, 8 loads in flight; FP64 sums in a fixed order.
// Bound by reading K_e, which the K D^{-1}F product before it has just read.
template <typename T, typename TU, int VW>
__global__ __launch_bounds__(256) void k_trace_rhs(int m, int n, const T* K, const TU* U, long su, double* Rh) {
  typedef T vecT __attribute__((ext_vector_type(VW)));
  constexpr int U8 = 8;
  __shared__ double red[4 * 64 * VW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long e = blockIdx.x;
  const T* Ke = K + e * static_cast<long>(m) * n;
  const TU* u = U + e * su;
  double* out = Rh + e * m;
  const int cper = (n + 3) / 4;
  const int c0 = wave * cper, c1 = min(n, c0 + cper);
  for (int r0 = 0; r0 < m; r0 += 64 * VW) {
    const int rows = min(64 * VW, m - r0);
    const int NL = rows / VW, G = 64 / NL;
    const int rg = lane % NL, cg = lane / NL;
    double acc[VW];
#pragma unroll
    for (int q = 0; q < VW; ++q) acc[q] = 0.0;
    if (cg < G) {
      const T* Kr = Ke + r0 + VW * rg;
      for (int cb = c0; cb < c1; cb += U8 * G) {
        vecT h[U8];
        double x[U8];
#pragma unroll
        for (int j = 0; j < U8; ++j) {
          const int c = min(cb + cg + G * j, c1 - 1);
          h[j] = *reinterpret_cast<const vecT*>(Kr + static_cast<long>(m) * c);
          x[j] = static_cast<double>(u[c]);
        }
#pragma unroll
        for (int j = 0; j < U8; ++j)
          if (cb + cg + G * j < c1)
#pragma unroll
            for (int q = 0; q < VW; ++q) acc[q] = fma(static_cast<double>(h[j][q]), x[j], acc[q]);
      }
#pragma unroll
      for (int q = 0; q < VW; ++q) red[(wave * G + cg) * rows + VW * rg + q] = acc[q];
    }
    __syncthreads();
    for (int t = tid; t < rows; t += 256) {
      double s = 0.0;
      for (int g = 0; g < 4 * G; ++g) s += red[g * rows + t];
      out[r0 + t] -= s;
    }
    __syncthreads();
  }
}

}  // namespace

template <typename T>
void matvec_elem(const Dims& d, const T* H, const TraceIn& in, double* we, hipStream_t s, const int* einst,
                 const double* emask) {
  products(Blocks{d.m, d.ncu, d.ndf, d.ne, einst, emask, nullptr}, H, in, we, s);
}

// x_f <- BE_f x_f of the block-Jacobi preconditioner (preconditioner.cpp:282-292): products of the faces' blocks
// with the faces' own nodes (one thread per row, reading a column at a time, 18 x 18 FP64, 10,800 faces: 12 us
// and 4.6 us for the gather before it; here 11.4 us with the gather)
template <typename T>
void bj_apply(const Dims& d, const T* BE, const TraceIn& in, double* y, hipStream_t s, const double* act) {
  products(Blocks{d.ncf, d.ncu, 0, d.nf, nullptr, nullptr, act}, BE, in, y, s);
}
template void bj_apply<double>(const Dims&, const double*, const TraceIn&, double*, hipStream_t, const double*);
template void bj_apply<float>(const Dims&, const float*, const TraceIn&, double*, hipStream_t, const double*);

template <typename T, typename TU>
void trace_rhs(const Dims& d, int eb, const T* K, const TU* U, long su, double* Rh, hipStream_t s) {
  if (eb <= 0) return;
  constexpr int VMAX = 16 / sizeof(T);
  if (d.m % VMAX == 0) k_trace_rhs<T, TU, VMAX><<<eb, 256, 0, s>>>(d.m, d.n, K, U, su, Rh);
  else if (d.m % 2 == 0) k_trace_rhs<T, TU, 2><<<eb, 256, 0, s>>>(d.m, d.n, K, U, su, Rh);
  else k_trace_rhs<T, TU, 1><<<eb, 256, 0, s>>>(d.m, d.n, K, U, su, Rh);
  EXA_HIP(hipGetLastError());
}

template void trace_rhs<double>(const Dims&, int, const double*, const double*, long, double*, hipStream_t);
template void trace_rhs<float>(const Dims&, int, const float*, const float*, long, double*, hipStream_t);
template void trace_rhs<float>(const Dims&, int, const float*, const double*, long, double*, hipStream_t);
template void matvec_elem<double>(const Dims&, const double*, const TraceIn&, double*, hipStream_t, const int*,
                                  const double*);
template void matvec_elem<float>(const Dims&, const float*, const TraceIn&, double*, hipStream_t, const int*,
                                 const double*);
template void matvec_elem<unsigned short>(const Dims&, const unsigned short*, const TraceIn&, double*, hipStream_t,
                                          const int*, const double*);

}  // namespace exa
