// bilu.hip -- the block-ILU(0) apply of small face blocks (ApplyBlockILU0,
// backend/Preconditioning/preconditioner.cpp:184-270).
#include "blkval.hpp"
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace exa {

namespace {

// Blocks of the program whose loads are in flight: about 64 registers of them, 8 at most
template <typename T, int VW, int CW>
constexpr int blocks_ahead() {
  const int regs = CW * ((static_cast<int>(sizeof(T)) * VW + 3) / 4);
  return regs >= 32 ? 2 : 64 / regs > 8 ? 8 : 64 / regs;
}

// One wave per superelement: lane (rr, part) accumulates rows VW rr .. VW rr + VW - 1 over columns
// CW part .. CW part + CW - 1 of every block.  The sweeps are one flat program of (block, vector offset)
// pairs in 3 nfse segments: forward rows 0 .. nfse-1, then for i = nfse-1 .. 0 the U row and the diagonal
// block, whose vector z lies after v.  A block of up to 32 rows is only a few loads per lane, so the sweep
// is a chain of load latencies unless several blocks are in flight: D of them are loaded ahead (no load
// waits for a row's result), and the program lies in LDS, read an entry ahead.  A segment's parts are added
// through LDS in a fixed order.
// ncf = 20 (2D Navier-Stokes, p = 4), BF16 factors, 1024 superelements of 2 x 2 quads: 33 us against 43 us
// with 256 threads and two barriers per row; what is left is the chain of row sums through LDS.
constexpr int PAD = 2 * 8 + 1;  // program entries read past its end: two rounds of 8 blocks and one

template <typename T, int VW, int CW>
__global__ __launch_bounds__(64) void k_bilu_apply_small(Dims d, IluDev I, const T* BE, const double* x, double* Xo,
                                                         const double* act) {
  if (act && act[0] == 0.0) return;  // a finished solve (grid-uniform)
  typedef T vecT __attribute__((ext_vector_type(VW)));
  using VT = typename std::conditional<sizeof(T) == 8, double, float>::type;  // as the general kernel's vector
  constexpr int D = blocks_ahead<T, VW, CW>();
  const int ncf = d.ncf, nfse = I.nfse;
  const int nrow = ncf / VW, nparts = 64 / nrow;
  const long n = blockIdx.x;
  const long per = static_cast<long>(ncf) * ncf, bstride = static_cast<long>(I.nse) * per;
  const int lane = threadIdx.x;
  const int rr = lane % nrow, part = lane / nrow;
  const int r0 = VW * rr;
  const bool active = part < nparts;
  const int c0 = active ? min(CW * part, ncf) : ncf;
  extern __shared__ double sm[];
  double* red = sm;                               // nparts ncf <= 64 VW
  int* pblk = reinterpret_cast<int*>(sm + 64 * VW);  // the program, repeating its last block: nprog + PAD each
  int* pvec = pblk + I.nprog + PAD;
  int* pseg = pvec + I.nprog + PAD;  // 3 nfse + 1 ends of segments
  VT* v = reinterpret_cast<VT*>(sm + 64 * VW + I.nprog + PAD + (3 * nfse + 2) / 2);  // nfse ncf, then z (ncf)
  for (int idx = lane; idx <= 3 * nfse; idx += 64) pseg[idx] = I.wseg[idx];
  for (int idx = lane; idx < I.nprog + PAD; idx += 64) {
    pblk[idx] = I.wblk[min(idx, I.nprog - 1)];
    pvec[idx] = I.wvec[min(idx, I.nprog - 1)];
  }
  for (int idx = lane; idx < nfse * ncf; idx += 64) {
    const int i = idx / ncf, q = idx % ncf;
    v[idx] = static_cast<VT>(x[static_cast<long>(I.face[n + static_cast<long>(I.nse) * i]) * ncf + q]);
  }
  __syncthreads();
  // the lane's columns (past the end: the last one, unused)
  int off[CW];
#pragma unroll
  for (int u = 0; u < CW; ++u) off[u] = ncf * min(c0 + u, ncf - 1) + r0;
  const T* base = BE + n * per;
  const int nseg = 3 * nfse;
  const int total = I.nprog;  // blocks in the program
  int sg = 0, send = pseg[1], send2 = pseg[min(2, nseg)];  // ends of this segment and the next
  double acc[VW];
#pragma unroll
  for (int j = 0; j < VW; ++j) acc[j] = 0.0;
  vecT raw[D][CW];
  auto issue = [&](int blk, vecT (&r)[CW]) {
    const T* p = base + __builtin_amdgcn_readfirstlane(blk) * bstride;
#pragma unroll
    for (int u = 0; u < CW; ++u) r[u] = *reinterpret_cast<const vecT*>(p + off[u]);
  };
  // segment sg is complete: add the parts and store its row's result
  auto finish = [&]() {
    if (active)
#pragma unroll
      for (int j = 0; j < VW; ++j) red[part * ncf + r0 + j] = acc[j];
#pragma unroll
    for (int j = 0; j < VW; ++j) acc[j] = 0.0;
    const int kind = sg < nfse ? 0 : 1 + ((sg - nfse) & 1);
    const int row = sg < nfse ? sg : nfse - 1 - (sg - nfse) / 2;
    if (lane < ncf) {
      double tot = 0.0;
      for (int p0 = 0; p0 < nparts; p0 += 8) {  // eight reads in flight, added in order
        double t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = red[min(p0 + u, nparts - 1) * ncf + lane];
#pragma unroll
        for (int u = 0; u < 8; ++u) tot += p0 + u < nparts ? t[u] : 0.0;
      }
      VT* vi = v + row * ncf + lane;
      VT* zi = v + nfse * ncf + lane;
      if (kind == 0) *vi = static_cast<VT>(static_cast<double>(*vi) - tot);
      else if (kind == 1) *zi = static_cast<VT>(static_cast<double>(*vi) - tot);
      else *vi = static_cast<VT>(tot);
    }
    __builtin_amdgcn_wave_barrier();
  };
  auto finish_through = [&](int q) {  // every segment that ends at or before block q
    while (sg < nseg && send <= q) {
      finish();
      ++sg;
      send = send2;
      send2 = pseg[min(sg + 2, nseg)];
    }
  };
  auto consume = [&](int q, int vec, const vecT (&r)[CW]) {
    const VT* y = v + vec + c0;
#pragma unroll
    for (int u = 0; u < CW; ++u)
      if (c0 + u < ncf) {
        const double yc = static_cast<double>(y[u]);
#pragma unroll
        for (int j = 0; j < VW; ++j) acc[j] = fma(blk_val<T>(r[u][j]), yc, acc[j]);
      }
    finish_through(q + 1);
  };
  finish_through(0);  // segments with no blocks before the first one
#pragma unroll
  for (int k = 0; k < D; ++k) issue(pblk[k], raw[k]);
  int bnext = pblk[D], vnext = pvec[0];
  // (past the last block the steps reread it and add to sums that no segment takes)
  for (int q = 0; q < total; q += D) {
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const int vec = vnext, blk = bnext;
      vnext = pvec[q + k + 1];
      bnext = pblk[q + k + D + 1];
      consume(q + k, vec, raw[k]);
      issue(blk, raw[k]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();
  for (int idx = lane; idx < nfse * ncf; idx += 64) {
    const int i = idx / ncf, q = idx % ncf;
    Xo[(n + static_cast<long>(I.nse) * i) * ncf + q] = v[idx];
  }
}

size_t small_lds(int ncf, int bytes, int nfse, int nprog, int VW) {
  return (64 * VW + nprog + PAD + (3 * nfse + 2) / 2) * sizeof(double) +
         static_cast<size_t>(nfse + 1) * ncf * (bytes == 8 ? sizeof(double) : sizeof(float));
}

template <typename T, int VW>
void apply_small_vw(const Dims& d, const IluDev& I, const T* BE, const double* x, double* Xo, const double* act, int cw,
                    hipStream_t s) {
  const size_t shm = small_lds(d.ncf, sizeof(T), I.nfse, I.nprog, VW);
  const auto go = [&](auto kern) { kern<<<I.nse, 64, shm, s>>>(d, I, BE, x, Xo, act); };
  if (cw == 1) go(&k_bilu_apply_small<T, VW, 1>);
  else if (cw == 2) go(&k_bilu_apply_small<T, VW, 2>);
  else if (cw == 3) go(&k_bilu_apply_small<T, VW, 3>);
  else if (cw == 4) go(&k_bilu_apply_small<T, VW, 4>);
  else if (cw <= 6) go(&k_bilu_apply_small<T, VW, 6>);
  else go(&k_bilu_apply_small<T, VW, 8>);
}

}  // namespace

// Time per apply with 256 threads / one wave (us), FP64, FP32 and BF16 factors, the scatter with it:
//   1 to 6 columns a lane: ncf 2 to 8, 1.6 to 2.5 times as fast; 9, 12, 16, 18: 1.2 to 2.4; 20, 24: 1.02 to 2.0
//   (2D and 3D superelements of 2 to 4 elements a side, 27 to 4,096 of them);
//   7 columns, ncf 28, 2D: 61/58 58/54 59/53 (512 of 2 x 2), 149/149 132/86 96/64 (2,048), 182/186 170/173 172/162 (128
//   of 4 x 4);
//   8 columns, ncf 32: 180/202 171/187 169/170 (27 of 2 x 2 x 2), 246/242 171/188 170/177 (216), 279/257 210/213 193/188
//   (512), 390/408 259/246 234/220 (1,000), 1730/1731 1293/1489 1208/1303 (64 of 4 x 4 x 4); 2D 48/50 52/50 52/49 (32 of
//   2 x 2), 61/59 56/53 56/52 (512), 186/194 140/108 96/74 (2,048), 165/183 164/172 163/162 (128 of 4 x 4), 251/231
//   201/195 180/169 (512).
// So: up to 7 columns always; 8, where few blocks fit the registers ahead, in FP32 and BF16 from 512 superelements.
int bilu_small_columns(int ncf, int bytes, int nse, int nfse, int nprog) {
  const int VW = ncf % 2 == 0 ? 2 : 1;
  if (ncf / VW > 64) return 0;
  const int nparts = 64 / (ncf / VW), cw = (ncf + nparts - 1) / nparts;
  if (cw > 8 || (cw == 8 && (bytes == 8 || nse < 512))) return 0;
  return small_lds(ncf, bytes, nfse, nprog, VW) <= 64 * 1024 ? cw : 0;
}

template <typename T>
bool bilu_apply_small(const Dims& d, const IluDev& I, const T* BE, const double* x, double* Xo, const double* act,
                      hipStream_t s) {
  const int cw = I.wseg ? bilu_small_columns(d.ncf, sizeof(T), I.nse, I.nfse, I.nprog) : 0;
  if (cw == 0) return false;
  if (d.ncf % 2 == 0) apply_small_vw<T, 2>(d, I, BE, x, Xo, act, cw, s);
  else apply_small_vw<T, 1>(d, I, BE, x, Xo, act, cw, s);
  return true;
}
template bool bilu_apply_small<double>(const Dims&, const IluDev&, const double*, const double*, double*,
                                       const double*, hipStream_t);
template bool bilu_apply_small<float>(const Dims&, const IluDev&, const float*, const double*, double*, const double*,
                                      hipStream_t);
template bool bilu_apply_small<unsigned short>(const Dims&, const IluDev&, const unsigned short*, const double*,
                                               double*, const double*, hipStream_t);

}  // namespace exa
