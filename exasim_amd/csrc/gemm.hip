// gemm.hip -- batched GEMMs of the assembly, the condensation LU and the set-up (strided batches
// of small dense products, uequation.cpp:559-775's schurMatrix* / the reference's batched BLAS
// calls) on gfx950, and the tile autotuner that picks each product's workgroup tile by measurement.
//
// Every product runs on the matrix cores (v_mfma_f64_16x16x4f64, or v_mfma_f32_16x16x4f32 for FP32
// products) with one of five workgroup tiles (BM x BN = 64x64, 32x64, 64x32, 128x64, 64x128), made of
// independent waves.  Every tile runs the same MFMA instruction over the same K order for each
// output element, so the tiles give bitwise-identical results and differ only in speed: the tuner
// times them on the first call of a product shape -- (M, N, K, the batch count's power of two,
// FP32 or FP64 products) -- on the caller's own operands (an accumulating product writes into a
// scratch copy of its C while it is timed), keeps the fastest for the process and launches it from
// then on.  No counterpart in the reference (its batched GEMMs are library calls).
#include "kernels.hpp"
#include "common.hpp"

#include <algorithm>
#include <array>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <type_traits>
#include <vector>

namespace exa {

namespace {

// ---------------------------------------------------------------------------
// Batched GEMM on the matrix cores, operands straight from global memory.
//
// Each wave computes FM x FN MFMA tiles of 16 x 16 by itself: no LDS, no barrier.  A 16-deep K block
// of both operands is held in registers while the next one's loads are in flight; the waves of one
// product run side by side and share operands through the caches.  Lane l of a 16x16x4 step supplies
// A[l%16][k] and B[k][l%16] with k = l/16 of the step; since a product's sum may take its K values in
// any order, step s of a block uses k = 4 (l/16) + s, so that a lane's four B values are contiguous
// and load as one vector.
//
// Bound by MFMA issue at the clock that the power limit leaves (counters of the 250 x 275 x 375 FP64
// product: the matrix cores busy 71 % of the cycles at 1.9 GHz), small K by the traffic of C.  Against
// the form with K tiles staged through LDS between two barriers, each on its best tile:
//   250 x 275 x 375, batch 2400:   FP64 3.77 -> 2.72 ms (33 -> 46 TFLOP/s), FP32 1.99 -> 1.67 ms (62 -> 74)
//   300 x 300 x 250, batch 1200:   FP64 1.94 -> 1.38 ms, FP32 1.10 -> 0.82 ms
//   186 x 487 x 64, batch 1200:    FP32 0.47 -> 0.40 ms (reads and writes C)
//   all updates of one FP64 LU, K = 32, n = 250, batch 2670 / batch 1200 / n = 196, batch 1000 / n = 64, batch 1331
//                                  9.95 -> 9.93 ms / 4.54 -> 4.26 / 1.13 -> 0.96 / 65 -> 54 us (read and write C)
//   144 x 36 x 72, batch 8100:     FP64 0.62 -> 0.40 ms, FP32 0.35 -> 0.20 ms
//   25 x 25 x 25, batch 25000:     FP64 117 -> 70 us
// ---------------------------------------------------------------------------
typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));
constexpr int KB = 16;  // K block

// One 16x16x4 step.  FP64: register i of lane l holds D[l/16 + 4i][l%16]; FP32: D[4(l/16) + i][l%16].
__device__ __forceinline__ dbl4 mfma_step(double a, double b, dbl4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ flt4 mfma_step(float a, float b, flt4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// A lane's four registers of an output tile hold pieces of W consecutive rows, piece h of lane l at row
// 4 W h + W (l/16) of the tile.  The matrix row that row r of the A operand's tile holds for this:
template <int W>
__device__ __forceinline__ int a_row(double, int r) {
  return W == 4 ? 4 * (r & 3) + (r >> 2) : 8 * (r >> 3) + 2 * (r & 3) + ((r >> 2) & 1);
}
template <int W>
__device__ __forceinline__ int a_row(float, int r) { return r; }

// W consecutive values at the alignment of one (global loads need no more)
template <typename T, int W> struct Vec;
template <int W> struct Vec<double, W> {
  typedef double type __attribute__((ext_vector_type(W), aligned(8)));
};
template <int W> struct Vec<float, W> {
  typedef float type __attribute__((ext_vector_type(W), aligned(4)));
};

// operands in the product's type
template <typename T> __device__ __forceinline__ T* gsel(double* d, float* f);
template <> __device__ __forceinline__ double* gsel<double>(double* d, float*) { return d; }
template <> __device__ __forceinline__ float* gsel<float>(double*, float* f) { return f; }
template <typename T> __device__ __forceinline__ const T* gsel(const double* d, const float* f);
template <> __device__ __forceinline__ const double* gsel<double>(const double* d, const float*) { return d; }
template <> __device__ __forceinline__ const float* gsel<float>(const double*, const float* f) { return f; }

// Workgroup w is dispatched to XCD w % 8 (each XCD has its own L2).  The logical
// id (w % 8) * (nwg / 8) + w / 8 gives every XCD a contiguous range of tiles,
// which run over the M/N tiles of one batch entry before the next, so the tiles
// that share an operand run together on one XCD and reuse it from its L2.
constexpr int NXCD = 8;

// Rows of a piece (W above).  In FP64 a lane's four rows lie together, 32 bytes, or in two pieces of 16, of which
// one access of the four lane groups covers 64 contiguous bytes of a column, where else its two accesses each take
// every other 16.  The small tile, which products bound by C run on, gains: 218 x 519 x 32, batch 2699, 1718 ->
// 1572 us; 154 x 455 x 32 1116 -> 1031; 90 x 391 x 32 614 -> 567.  The larger ones, with C read after the K loop, lose
// (four rows / two pieces): 4 x 4 MFMA tiles 1964/2467, 4 x 2 1999/1994, 2 x 4 1990/2094 us in the first.
template <typename T, int FM, int FN>
constexpr int rows_piece() { return sizeof(T) == 8 && FM * FN <= 4 ? 2 : 4; }

// A workgroup of WM x WN waves; T: double or float throughout.  Two waves per SIMD (256 registers),
// except for the FP64 4 x 4 tiles, whose accumulators and operand blocks take more.
template <typename T, int FM, int FN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN)
__attribute__((amdgpu_waves_per_eu(sizeof(T) * FM * FN > 64 ? 1 : 2)))
void k_gemm(Gemm g, int tilesM, int tilesN, unsigned ntiles) {
  constexpr int W = rows_piece<T, FM, FN>(), NP = 4 / W, STEP = 4 * W;
  typedef typename Vec<T, 4>::type v4;
  typedef typename Vec<T, W>::type piece;
  typedef T acc4 __attribute__((ext_vector_type(4)));
  const unsigned nwg = gridDim.x;  // a multiple of NXCD
  const unsigned L = (blockIdx.x % NXCD) * (nwg / NXCD) + blockIdx.x / NXCD;
  if (L >= ntiles) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned tpb = tilesM * tilesN;
  const unsigned b = L / tpb, tt = L - b * tpb;
  const unsigned b0 = b % static_cast<unsigned>(g.nb0), t1 = b / static_cast<unsigned>(g.nb0);
  const unsigned b1 = t1 % static_cast<unsigned>(g.nb1), b2 = t1 / static_cast<unsigned>(g.nb1);
  const int M = g.M, N = g.N, K = g.K;
  const int row0 = (tt % tilesM * WM + wave % WM) * (16 * FM), col0 = (tt / tilesM * WN + wave / WM) * (16 * FN);
  if (row0 >= M || col0 >= N) return;
  const long a0 = g.iA ? g.iA[b0] : b0, bb0 = g.iB ? g.iB[b0] : b0, c0 = g.iC ? g.iC[b0] : b0;
  const T* A = gsel<T>(g.A, g.Af) + g.sA0 * a0 + g.sA1 * b1 + g.sA2 * b2;
  const T* B = gsel<T>(g.B, g.Bf) + g.sB0 * bb0 + g.sB1 * b1 + g.sB2 * b2;
  T* C = gsel<T>(g.C, g.Cf) + g.sC0 * c0 + g.sC1 * b1 + g.sC2 * b2;
  const int li = lane & 15, lk = lane >> 4;
  // Byte offsets of the lane's rows of A and columns of B, 32 bits each beside a uniform base.  Rows and
  // columns past the end read the last one; their results are not written.
  const unsigned lda = static_cast<unsigned>(g.lda);
  const unsigned ka = lda * (4 * lk), kb = 4 * lk;
  unsigned oa[FM], ob[FN];
#pragma unroll
  for (int i = 0; i < FM; ++i) oa[i] = (min(row0 + 16 * i + a_row<W>(T(0), li), M - 1) + ka) * sizeof(T);
#pragma unroll
  for (int j = 0; j < FN; ++j)
    ob[j] = (static_cast<unsigned>(g.ldb) * min(col0 + 16 * j + li, N - 1) + kb) * sizeof(T);
  auto at_byte = [](const T* base, unsigned off) { return reinterpret_cast<const char*>(base) + off; };
  acc4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = acc4{0, 0, 0, 0};
  // MFMA tiles of the wave that hold output (the others' loads are harmless, their products skipped)
  const int fm = min(FM, (M - row0 + 15) / 16), fn = min(FN, (N - col0 + 15) / 16);
  T av[2][FM][4];
  v4 bv[2][FN];
  auto load = [&](int buf, int k0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const T* Ak = A + g.lda * (k0 + s);
#pragma unroll
      for (int i = 0; i < FM; ++i) av[buf][i][s] = *reinterpret_cast<const T*>(at_byte(Ak, oa[i]));
    }
    const T* Bk = B + k0;
#pragma unroll
    for (int j = 0; j < FN; ++j) bv[buf][j] = *reinterpret_cast<const v4*>(at_byte(Bk, ob[j]));
  };
  // the products of the block in buffer buf, interleaved with the loads of the next one into the
  // other (one load after every few products keeps both queues fed)
  auto block = [&](int buf, int knext) {
    load(buf ^ 1, knext);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma_step(av[buf][i][s], bv[buf][j][s], acc[i][j]);
    constexpr int NLOAD = 4 * FM + FN * (sizeof(T) == 8 ? 2 : 1), PER = 4 * FM * FN / NLOAD;
#pragma unroll
    for (int q = 0; q < NLOAD; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);   // one global load
      __builtin_amdgcn_sched_group_barrier(0x8, PER, 0);  // PER products
    }
    __builtin_amdgcn_sched_group_barrier(0x8, 4 * FM * FN - PER * NLOAD, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // the same for a wave whose last MFMA tiles lie past the matrix: their products are skipped
  auto block_edge = [&](int buf, int knext) {
    load(buf ^ 1, knext);
#pragma unroll
    for (int j = 0; j < FN; ++j)
      if (j < fn)
#pragma unroll
        for (int i = 0; i < FM; ++i)
          if (i < fm)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[i][j] = mfma_step(av[buf][i][s], bv[buf][j][s], acc[i][j]);
  };
  // an accumulating product's C, read before the K loop where the registers allow (with few K blocks
  // its latency would otherwise follow theirs)
  constexpr bool EARLY_C = sizeof(T) * FM * FN <= 32;
  const T alpha = static_cast<T>(g.alpha), beta = static_cast<T>(g.beta);
  piece cv[FM][FN][NP];
  auto load_c = [&](int i, int j, int h) {
    const int r = row0 + 16 * i + STEP * h + W * lk, c = col0 + 16 * j + li;
    if (c < N && r + W <= M) cv[i][j][h] = *reinterpret_cast<const piece*>(C + r + g.ldc * c);
  };
  if (EARLY_C && beta != T(0)) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int h = 0; h < NP; ++h) load_c(i, j, h);
  }
  // A block's loads are always issued (past the end: the last block again, unused), so that the wait
  // before the products counts only older loads.
  const int nk = K / KB;
  if (nk > 0) {
    load(0, 0);
    int t = 0;
    if (fm == FM && fn == FN) {
      for (; t + 2 <= nk; t += 2) {
        block(0, KB * (t + 1));
        block(1, KB * min(t + 2, nk - 1));
      }
      if (t < nk) block(0, KB * t);
    } else {
      for (; t + 2 <= nk; t += 2) {
        block_edge(0, KB * (t + 1));
        block_edge(1, KB * min(t + 2, nk - 1));
      }
      if (t < nk) block_edge(0, KB * t);
    }
  }
  // the last K % 16 values, 4 per step (k = l/16 of the step; zeros past K)
  const int kt = nk * KB;
  if (kt < K) {
    T at[4][FM], bt[4][FN];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (kt + 4 * s < K) {
        const int k = kt + 4 * s + lk, kc = min(k, K - 1);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const T x = *reinterpret_cast<const T*>(at_byte(A, oa[i] + (lda * kc - ka) * unsigned(sizeof(T))));
          at[s][i] = k < K ? x : T(0);
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const T x = *reinterpret_cast<const T*>(at_byte(B, ob[j] + (kc - kb) * unsigned(sizeof(T))));
          bt[s][j] = k < K ? x : T(0);
        }
      }
#pragma unroll
    for (int s = 0; s < 4; ++s)
      if (kt + 4 * s < K)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] = mfma_step(at[s][i], bt[s][j], acc[i][j]);
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int h = 0; h < NP; ++h) {
        const int r = row0 + 16 * i + STEP * h + W * lk, c = col0 + 16 * j + li;
        if (c >= N || r >= M) continue;
        T* p = C + r + g.ldc * c;
        if (r + W <= M) {
          piece x;
          if (beta != T(0)) {
            if (!EARLY_C) load_c(i, j, h);
#pragma unroll
            for (int q = 0; q < W; ++q) x[q] = fma(beta, cv[i][j][h][q], alpha * acc[i][j][W * h + q]);
          } else {
#pragma unroll
            for (int q = 0; q < W; ++q) x[q] = alpha * acc[i][j][W * h + q];
          }
          *reinterpret_cast<piece*>(p) = x;
        } else {
#pragma unroll
          for (int q = 0; q < W - 1; ++q)
            if (r + q < M) {
              const T v = alpha * acc[i][j][W * h + q];
              p[q] = beta != T(0) ? fma(beta, p[q], v) : v;
            }
        }
      }
}

// ---------------------------------------------------------------------------
// Launchers: one per (type, tile).  wrows, wcols: the rows and columns of a tile that one wave holds.
// ---------------------------------------------------------------------------
struct TileShape {
  int bm, bn, wrows, wcols;
};
constexpr int NTILE = 5;
constexpr TileShape TILES[NTILE] = {{64, 64, 64, 64}, {32, 64, 32, 32}, {64, 32, 64, 32}, {128, 64, 64, 32},
                                    {64, 128, 32, 64}};

typedef void (*MfmaLaunch)(const Gemm&, hipStream_t);

template <typename T, int FM, int FN, int WM, int WN>
void launch_mfma(const Gemm& g, hipStream_t s) {
  constexpr int BM = 16 * FM * WM, BN = 16 * FN * WN;
  const long batch = static_cast<long>(g.nb0) * g.nb1 * g.nb2;
  const int tm = (g.M + BM - 1) / BM, tn = (g.N + BN - 1) / BN;
  const long ntiles = static_cast<long>(tm) * tn * batch;
  const long nwg = (ntiles + NXCD - 1) / NXCD * NXCD;
  if (nwg > 0x7fffffffL) throw Error(5, "GEMM batch too large for one launch");
  k_gemm<T, FM, FN, WM, WN><<<static_cast<unsigned>(nwg), 64 * WM * WN, 0, s>>>(g, tm, tn,
                                                                                 static_cast<unsigned>(ntiles));
}

template <typename T>
constexpr std::array<MfmaLaunch, NTILE> tile_launchers() {
  return {launch_mfma<T, 4, 4, 1, 1>, launch_mfma<T, 2, 2, 1, 2>, launch_mfma<T, 4, 2, 1, 1>,
          launch_mfma<T, 4, 2, 2, 2>, launch_mfma<T, 2, 4, 2, 2>};
}

MfmaLaunch mfma_launcher(int fp32, int tile) {
  static constexpr auto f64 = tile_launchers<double>();
  static constexpr auto f32 = tile_launchers<float>();
  return fp32 ? f32[tile] : f64[tile];
}

// ---------------------------------------------------------------------------
// The elimination of q from the trace rows, K = K0 + G M^-1 C and H = H0 - G M^-1 E, for the eb elements
// of a block.  A trace row of face l couples only with the q nodes on that face, so its products run over
// the npf nd rows of M^-1 C and M^-1 E at the face's nodes (frow) instead of all npe nd, with G stored
// without its zeros: G[t + m (j + npf d + npf nd c)], t = k + ncu (i + npf l) a trace row, j the face node, d, c
// the direction and component of q.  K0 = K0c[t + m (j + npf c)] and H0 = H0c[t + m (c + ncu j)] lie at the
// face's own nodes (finv: face node of an element node, or -1) and are added where they are, so that K
// and H are written once and read by nothing before.
//
// Bound by MFMA issue and the writes of K and H.  One workgroup per element and 16 FN columns of
// M^-1 C or M^-1 E, which are staged in LDS once (STAGE) and serve every face and component: the rows a
// face gathers lie far apart in global memory (read from there, each load touched up to 64 cache lines: 20^3
// hexes, p = 4, two components, 15.4 ms FP64 and 10.3 ms FP32 per assembly against 11.8 and 7.1).  A wave takes FM x FN MFMA tiles of a (face, component) pair at a time, G straight
// from global memory a 16-deep block ahead.  The dense products it replaces needed 3.9 times the MFMAs
// there, and G, K and H cleared first.
// ---------------------------------------------------------------------------
template <typename T, int FM, int FN, bool STAGE>
__global__ __launch_bounds__(256) void k_face_elim(FaceElim<T> f, int kpad, int tilesM, int tilesK, int tilesH) {
  constexpr int W = 16 / sizeof(T), NP = 4 / W, STEP = 4 * W;  // as k_gemm's small tiles
  typedef typename Vec<T, W>::type piece;
  typedef T acc4 __attribute__((ext_vector_type(4)));
  extern __shared__ double face_sm[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int ncu = f.ncu, npf = f.npf, npe = f.npe, nd = f.nd, nfe = f.nfe, m = f.m;
  const int M = ncu * npf, K = npf * nd, ndf = npf * nfe, ldb = npe * nd;
  const int ldl = ldb | 1;  // column stride in LDS: odd, so that 16 columns meet different banks
  const unsigned tiles = tilesK + tilesH;
  const unsigned nwg = gridDim.x;  // a multiple of NXCD
  const unsigned L = (blockIdx.x % NXCD) * (nwg / NXCD) + blockIdx.x / NXCD;
  if (L >= tiles * static_cast<unsigned>(f.eb)) return;
  const long e = L / tiles;
  const int tcol = L % tiles;
  const bool isH = tcol >= tilesK;
  const int N = isH ? ndf : npe;
  const int col0 = (isH ? tcol - tilesK : tcol) * (16 * FN);
  const T* B = isH ? f.ME + (f.e0 + e) * static_cast<long>(ldb) * ndf : f.MC + (f.e0 + e) * static_cast<long>(ldb) * npe;
  int* rows = reinterpret_cast<int*>(face_sm);  // [nfe][kpad]: rows of M^-1 C / M^-1 E, K of them and zeros
  T* Bs = reinterpret_cast<T*>(face_sm + (nfe * kpad + 1) / 2);  // [16 FN][ldl]
  for (int l = wave; l < nfe; l += 4)
    for (int k = lane; k < kpad; k += 64) rows[l * kpad + k] = k < K ? f.frow[l * K + k] : 0;
  if (STAGE)
    for (int c = wave; c < 16 * FN && col0 + c < N; c += 4) {
      const T* Bc = B + static_cast<long>(ldb) * (col0 + c);
      for (int r = lane; r < ldb; r += 64) Bs[c * ldl + r] = Bc[r];
    }
  __syncthreads();
  // columns past the end read the last one; their results are not written
  unsigned ob[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int c = min(col0 + 16 * j + li, N - 1);
    ob[j] = STAGE ? (c - col0) * ldl : static_cast<unsigned>(ldb) * c;
  }
  const unsigned lda = static_cast<unsigned>(m) * unsigned(sizeof(T));
  for (int task = wave; task < nfe * ncu * tilesM; task += 4) {
    const int row0 = task % tilesM * (16 * FM), cp = task / tilesM % ncu, l = task / tilesM / ncu;
    const T* A = f.G + e * static_cast<long>(m) * K * ncu + static_cast<long>(m) * K * cp + l * M;
    unsigned oa[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) oa[i] = min(row0 + 16 * i + a_row<W>(T(0), li), M - 1) * unsigned(sizeof(T));
    acc4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = acc4{0, 0, 0, 0};
    T av[2][FM][4];
    auto load = [&](int buf, int k0) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const char* Ak = reinterpret_cast<const char*>(A) + lda * min(k0 + 4 * lk + s, K - 1);
#pragma unroll
        for (int i = 0; i < FM; ++i) av[buf][i][s] = *reinterpret_cast<const T*>(Ak + oa[i]);
      }
    };
    auto products = [&](int buf, int k0) {
      const int4 r = *reinterpret_cast<const int4*>(rows + l * kpad + k0 + 4 * lk);
      const int rr[4] = {r.x, r.y, r.z, r.w};
      T bv[FN][4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < FN; ++j) bv[j][s] = STAGE ? Bs[ob[j] + rr[s]] : B[ob[j] + rr[s]];
      if (k0 + KB > K)  // values past K count as zeros in both operands
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const bool ok = k0 + 4 * lk + s < K;
#pragma unroll
          for (int i = 0; i < FM; ++i) av[buf][i][s] = ok ? av[buf][i][s] : T(0);
#pragma unroll
          for (int j = 0; j < FN; ++j) bv[j][s] = ok ? bv[j][s] : T(0);
        }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] = mfma_step(av[buf][i][s], bv[j][s], acc[i][j]);
    };
    // kpad is K rounded up to whole 16-deep blocks; a block past the end reads the last one, unused
    load(0, 0);
    for (int k0 = 0; k0 < kpad; k0 += 2 * KB) {
      load(1, min(k0 + KB, kpad - KB));
      products(0, k0);
      if (k0 + KB >= kpad) break;
      load(0, min(k0 + 2 * KB, kpad - KB));
      products(1, k0 + KB);
    }
    T* C = isH ? f.H + (f.e0 + e) * static_cast<long>(m) * m : f.K + e * static_cast<long>(m) * f.n;
    const T* X = isH ? f.H0c + e * static_cast<long>(m) * M : f.K0c + e * static_cast<long>(m) * M;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int c = col0 + 16 * j + li;
      if (c >= N) continue;
      long at, x0 = -1;  // column of K or H, and of its face-node part
      if (isH) {
        at = cp + ncu * c;
        if (c / npf == l) x0 = cp + ncu * (c - npf * l);
      } else {
        at = c + npe * cp;
        const int v = f.finv[l * npe + c];
        if (v >= 0) x0 = v + npf * cp;
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int h = 0; h < NP; ++h) {
          const int r = row0 + 16 * i + STEP * h + W * lk;
          T* p = C + m * at + l * M + r;
          const T* x = X + m * max(x0, 0L) + l * M + r;
          piece v;
#pragma unroll
          for (int t = 0; t < W; ++t) {
            const T y = acc[i][j][W * h + t];
            v[t] = isH ? -y : y;
            if (x0 >= 0 && r + t < M) v[t] += x[t];
          }
          if (r + W <= M) *reinterpret_cast<piece*>(p) = v;
          else
#pragma unroll
            for (int t = 0; t < W - 1; ++t)
              if (r + t < M) p[t] = v[t];
        }
    }
  }
}

template <typename T, int FM, int FN, bool STAGE>
void launch_face_elim(const FaceElim<T>& f, size_t lds, hipStream_t s) {
  const int M = f.ncu * f.npf, kpad = (f.npf * f.nd + KB - 1) / KB * KB;
  const int tm = (M + 16 * FM - 1) / (16 * FM), tk = (f.npe + 16 * FN - 1) / (16 * FN),
            th = (f.npf * f.nfe + 16 * FN - 1) / (16 * FN);
  const long nwg = (static_cast<long>(tk + th) * f.eb + NXCD - 1) / NXCD * NXCD;
  if (nwg > 0x7fffffffL) throw Error(5, "element block too large for one launch");
  k_face_elim<T, FM, FN, STAGE><<<static_cast<unsigned>(nwg), 256, lds, s>>>(f, kpad, tm, tk, th);
}

// The columns of a workgroup: as many 16-column tiles (4, 2 or 1) as 56 KB of LDS hold, so that two
// workgroups or more share a CU; elements whose single tile takes more read M^-1 C and M^-1 E from memory.
template <typename T, int FM>
void face_elim_fm(const FaceElim<T>& f, hipStream_t s) {
  const int kpad = (f.npf * f.nd + KB - 1) / KB * KB;
  const size_t idx = static_cast<size_t>((f.nfe * kpad + 1) / 2) * sizeof(double);
  const size_t col16 = 16 * sizeof(T) * static_cast<size_t>(f.npe * f.nd | 1);
  constexpr size_t LIMIT = 56 * 1024;
  if (idx + 4 * col16 <= LIMIT) launch_face_elim<T, FM, 4, true>(f, idx + 4 * col16, s);
  else if (idx + 2 * col16 <= LIMIT) launch_face_elim<T, FM, 2, true>(f, idx + 2 * col16, s);
  else if (idx + col16 <= LIMIT) launch_face_elim<T, FM, 1, true>(f, idx + col16, s);
  else launch_face_elim<T, FM, 2, false>(f, idx, s);
}

// ---------------------------------------------------------------------------
// The autotuner
// ---------------------------------------------------------------------------
typedef std::tuple<int, int, int, int, int, int> TuneKey;  // device, M, N, K, log2 batch, fp32
struct TuneEntry {
  int tile = 0;
  long batch = 0;  // products in the timed call
  float us[NTILE] = {0};
};
std::mutex tune_mu;
std::map<TuneKey, TuneEntry>& tune_table() {
  static std::map<TuneKey, TuneEntry> t;
  return t;
}
int tune_mode() {  // 1: time the tiles on the first call of a shape; 0: the default tile
  static int m = [] {
    const char* e = std::getenv("EXA_GEMM_AUTOTUNE");
    return e ? std::atoi(e) : 1;
  }();
  return m;
}
int& tune_override() {  // set by set_gemm_autotune (-1: the environment's choice)
  static int v = -1;
  return v;
}
int& forced_tile() {  // set by set_gemm_tile: every MFMA product on this tile (-1: the tuner's)
  static int v = -1;
  return v;
}

int log2_bucket(long v) {
  int k = 0;
  while ((1L << (k + 1)) <= v) ++k;
  return k;
}

// A product may be run again on its own C for timing only when that leaves C as one run leaves
// it: beta = 0 and C apart from A and B (the tiles write identical values).
bool rerunnable(const Gemm& g) {
  if (g.beta != 0.0) return false;
  const void* c = g.Cf ? static_cast<const void*>(g.Cf) : static_cast<const void*>(g.C);
  const void* a = g.Af ? static_cast<const void*>(g.Af) : static_cast<const void*>(g.A);
  const void* b = g.Bf ? static_cast<const void*>(g.Bf) : static_cast<const void*>(g.B);
  return c != a && c != b;
}

// A product computed in place (C is B, as the LU's X = T^{-1} X) is correct only when one wave
// holds all rows of its columns (every row of B is read before any row of C is written);
// C is A likewise needs all columns in one wave.
bool tile_ok(const Gemm& g, int t) {
  const void* c = g.Cf ? static_cast<const void*>(g.Cf) : static_cast<const void*>(g.C);
  const void* a = g.Af ? static_cast<const void*>(g.Af) : static_cast<const void*>(g.A);
  const void* b = g.Bf ? static_cast<const void*>(g.Bf) : static_cast<const void*>(g.B);
  if (c == b && TILES[t].wrows < g.M) return false;
  if (c == a && TILES[t].wcols < g.N) return false;
  return true;
}

// Elements C spans (strided batches without an index map), or -1
long c_extent(const Gemm& g) {
  if (g.iC || g.sC0 < 0 || g.sC1 < 0 || g.sC2 < 0) return -1;
  return g.sC0 * (g.nb0 - 1) + g.sC1 * (g.nb1 - 1) + g.sC2 * (g.nb2 - 1) + g.ldc * static_cast<long>(g.N - 1) +
         g.M;
}

// the tile for this product: the table's, or timed now (every tile five times after one warm-up
// run, the fastest run kept, so that work of other streams inflates no tile's time), or the
// default when the shape cannot be timed.  A product that cannot be rerun on its own C is timed
// writing into a scratch copy of C's extent (its values are not used).
int pick_tile(const Gemm& g, long batch, hipStream_t s) {
  if (forced_tile() >= 0) return tile_ok(g, forced_tile()) ? forced_tile() : 0;
  const int mode = tune_override() >= 0 ? tune_override() : tune_mode();
  if (mode == 0) return 0;
  const long work = static_cast<long>((g.M + 63) / 64) * ((g.N + 63) / 64) * batch;
  if (work < 64) return tile_ok(g, 1) ? 1 : 0;  // a launch of a few workgroups: the smallest tile spreads widest
  int dev = 0;
  EXA_HIP(hipGetDevice(&dev));
  const TuneKey key{dev, g.M, g.N, g.K, log2_bucket(batch), g.fp32};
  {
    std::lock_guard<std::mutex> lk(tune_mu);
    auto it = tune_table().find(key);
    if (it != tune_table().end()) return tile_ok(g, it->second.tile) ? it->second.tile : 0;
  }
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  EXA_HIP(hipStreamIsCapturing(s, &cap));
  if (cap != hipStreamCaptureStatusNone) return 0;  // no timing inside a graph capture
  Gemm gt = g;
  void* scratch = nullptr;
  if (!rerunnable(g)) {
    const long ext = c_extent(g);
    const size_t bytes = static_cast<size_t>(ext) * (g.Cf ? sizeof(float) : sizeof(double));
    if (ext <= 0 || bytes > (size_t(4) << 30)) return 0;
    EXA_HIP(hipStreamSynchronize(s));
    if (hipMalloc(&scratch, bytes) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    EXA_HIP(hipMemsetAsync(scratch, 0, bytes, s));
    if (g.Cf) gt.Cf = static_cast<float*>(scratch);
    else gt.C = static_cast<double*>(scratch);
  }
  TuneEntry ent;
  ent.batch = batch;
  hipEvent_t e0, e1;
  EXA_HIP(hipEventCreate(&e0));
  EXA_HIP(hipEventCreate(&e1));
  float best = 0.0f;
  for (int t = 0; t < NTILE; ++t) {
    if (!tile_ok(g, t)) {
      ent.us[t] = -1.0f;  // not a candidate for this product
      continue;
    }
    const MfmaLaunch f = mfma_launcher(g.fp32, t);
    f(gt, s);  // warm-up
    float fastest = 0.0f;
    for (int r = 0; r < 5; ++r) {
      float ms = 0.0f;
      EXA_HIP(hipEventRecord(e0, s));
      f(gt, s);
      EXA_HIP(hipEventRecord(e1, s));
      EXA_HIP(hipEventSynchronize(e1));
      EXA_HIP(hipEventElapsedTime(&ms, e0, e1));
      if (r == 0 || ms < fastest) fastest = ms;
    }
    ent.us[t] = fastest * 1000.0f;
    if (t == 0 || ent.us[t] < best) {  // (tile 0 is always a candidate: in-place products have M, N <= 64)
      best = ent.us[t];
      ent.tile = t;
    }
  }
  EXA_HIP(hipEventDestroy(e0));
  EXA_HIP(hipEventDestroy(e1));
  if (scratch) {
    EXA_HIP(hipStreamSynchronize(s));
    EXA_HIP(hipFree(scratch));
  }
  EXA_HIP(hipGetLastError());
  std::lock_guard<std::mutex> lk(tune_mu);
  tune_table()[key] = ent;
  return ent.tile;
}

}  // namespace

void gemm(const Gemm& g, hipStream_t s) {
  if (g.M <= 0 || g.N <= 0) return;
  const long batch = static_cast<long>(g.nb0) * g.nb1 * g.nb2;
  if (batch <= 0) return;
  const int store = (g.Af ? 1 : 0) | (g.Bf ? 2 : 0) | (g.Cf ? 4 : 0);
  if (store != (g.fp32 ? 7 : 0)) throw Error(5, "GEMM operands must be stored in the product's type");
  // the scaling and the sum with C are exact up to the one rounding of the result for these
  if (g.fp32 && ((g.alpha != 1.0 && g.alpha != -1.0) || (g.beta != 0.0 && g.beta != 1.0)))
    throw Error(5, "FP32 GEMM coefficients must be alpha = 1 or -1, beta = 0 or 1");
  // the kernel's offsets within one A or B are 32-bit
  if (g.lda * static_cast<long>(g.K) + g.M > 0x1fffffffL || g.ldb * static_cast<long>(g.N) + g.K > 0x1fffffffL)
    throw Error(5, "GEMM operand too large");
  // products of at most one 32 x 32 tile run on it; the tuner picks the others' tile
  const int tile = g.M <= 32 && g.N <= 32 && forced_tile() < 0 ? 1 : pick_tile(g, batch, s);
  // (a product timed on its own C has left its result there; one more run writes the same values)
  mfma_launcher(g.fp32, tile)(g, s);
  EXA_HIP(hipGetLastError());
}

template <typename T>
void face_elim(const FaceElim<T>& f, hipStream_t s) {
  if (f.eb <= 0) return;
  // a wave's rows: one, two or four MFMA tiles, by the rows of a face
  const int M = f.ncu * f.npf;
  if (M <= 16) face_elim_fm<T, 1>(f, s);
  else if (M <= 32) face_elim_fm<T, 2>(f, s);
  else face_elim_fm<T, 4>(f, s);
  EXA_HIP(hipGetLastError());
}
template void face_elim<double>(const FaceElim<double>&, hipStream_t);
template void face_elim<float>(const FaceElim<float>&, hipStream_t);

void set_gemm_autotune(int mode) { tune_override() = mode; }

void set_gemm_tile(int tile) {
  if (tile < -1 || tile >= NTILE) throw Error(1, "gemm_tile: -1 (the tuner's choice) or 0..4");
  forced_tile() = tile;
}

std::string gemm_tuning_report() {
  std::lock_guard<std::mutex> lk(tune_mu);
  std::string out;
  char line[320];
  for (const auto& kv : tune_table()) {
    const TuneKey& k = kv.first;
    const TuneEntry& e = kv.second;
    const int fp32 = std::get<5>(k);  // the storage field: bits of the operands in FP32, all or none
    std::snprintf(line, sizeof line, "%d %d %d %d %d %d %dx%d %ld", std::get<1>(k), std::get<2>(k), std::get<3>(k),
                  std::get<4>(k), fp32, fp32 ? 7 : 0, TILES[e.tile].bm, TILES[e.tile].bn, e.batch);
    out += line;
    for (int t = 0; t < NTILE; ++t) {
      std::snprintf(line, sizeof line, " %.3f", e.us[t]);
      out += line;
    }
    out += "\n";
  }
  return out;
}

}  // namespace exa
