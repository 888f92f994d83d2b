// FP64 dense factorisations on the GPU for the K x K matrices of the path:
// Cholesky of CC^T and of V (pzpotrf 'L' in the reference,
// src/matrix_operations.h:259-267) and the SPD inverse used to apply
// CC^T^-1 to ZC^T as one MFMA GEMM.
//
// Cholesky: right-looking, 64-column panels, one fused kernel per panel
// (panel solve by the inverse of the diagonal block, trailing update, and the
// next diagonal block's factor and inverse); layout below.
// Inverse: the lower factor is padded with an identity to 64 * 2^p, its
// 64 x 64 diagonal blocks are inverted in parallel, then recursive doubling
// forms Linv21 = -Linv22 (L21 Linv11) for every pair of blocks of one size in
// two batched GEMMs per level; finally A^-1 = Linv^T Linv.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <utility>

#include "common.h"

namespace thc {
namespace {

constexpr int NB = 64;

// ---- fused right-looking Cholesky ------------------------------------------
// The matrix is taken in 64 x 64 blocks, extended by the identity beyond k.
// Step j (one kernel) owns panel j: its diagonal block was factored by step
// j - 1, which also left W_j = L_jj^-1.  Every workgroup takes one lower tile
// (I, J) of the trailing matrix (I >= J > j) and
//   1. forms L_I = A_Ij W_j^T and L_J = A_Jj W_j^T (MFMA, from the unsolved
//      panel rows, so the panel itself is never rewritten during the step);
//   2. applies A_IJ -= L_I L_J^T (MFMA);
//   3. for I = J, parks L_I transposed in the unused upper block (j, I);
//   4. tile (j+1, j+1) -- workgroup 0 -- then factors its block in panels of
//      16 columns (factor_block) and forms W_{j+1}.
// A last kernel moves the parked panels into the lower triangle and zeroes
// the upper one.  Step -1 only factors block 0.
constexpr int CB = NB;      // block size
constexpr int CT = 4 * 64;  // threads of a step workgroup

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ inline d4 mfma_f64(double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

__device__ inline double readlane_d(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// 1/sqrt(d) from the hardware reciprocal square root (about 23 bits) and two
// Newton steps y <- y (3/2 - d/2 y^2) (quadratic: 2^-23 -> 2^-45 -> rounding
// level), sqrt(d) = d / sqrt(d); seven dependent operations after the
// estimate.  Non-positive or NaN d give NaN, as sqrt would.
__device__ inline void sqrt_rsqrt(double d, double& s, double& rs) {
  const double h = 0.5 * d;
  double y = __builtin_amdgcn_rsq(d);
  y = y * fma(-h, y * y, 1.5);
  y = y * fma(-h, y * y, 1.5);
  rs = y;
  s = d * y;
}

// a[r][c] of the matrix extended by the identity beyond k
__device__ inline double ext_at(const double* a, long lda, int k, long r, long c) {
  const bool in = r < k && c < k;
  const double v = a[in ? r * lda + c : 0];
  return in ? v : (r == c ? 1.0 : 0.0);
}

// Block at (r0, c0) into X; each wave reads whole 64-element rows, all loads
// issued before the first LDS store.
__device__ inline void load_tile(const double* a, long lda, int k, long r0, long c0, double (*X)[CB + 1]) {
  const int c = threadIdx.x & 63, rb = threadIdx.x >> 6;
  double v[CB / 4];
#pragma unroll
  for (int i = 0; i < CB / 4; ++i) v[i] = ext_at(a, lda, k, r0 + rb + 4 * i, c0 + c);
#pragma unroll
  for (int i = 0; i < CB / 4; ++i) X[rb + 4 * i][c] = v[i];
}

// Rows 16 w .. 16 w + 15 of X become X W^T (wave w; only its own rows are
// read and then rewritten).  wf: fragments of W, which is lower triangular, so
// that wf[q][cb] is read for 16 cb + 15 >= 4 q only.  f64 MFMA D layout: lane
// l holds column l % 16 of rows l / 16 + 4 v.
__device__ __forceinline__ void panel_rows(double (*X)[CB + 1], const double (&wf)[CB / 4][4]) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  d4 acc[4] = {};
  double af[CB / 4];
#pragma unroll
  for (int q = 0; q < CB / 4; ++q) af[q] = X[16 * w + (l & 15)][4 * q + (l >> 4)];
#pragma unroll
  for (int q = 0; q < CB / 4; ++q)
#pragma unroll
    for (int cb = q / 4; cb < 4; ++cb) acc[cb] = mfma_f64(af[q], wf[q][cb], acc[cb]);
#pragma unroll
  for (int cb = 0; cb < 4; ++cb)
#pragma unroll
    for (int v = 0; v < 4; ++v) X[16 * w + (l >> 4) + 4 * v][16 * cb + (l & 15)] = acc[cb][v];
}

// ---- 64 x 64 block factor and inverse ---------------------------------------
// Both work in panels of PB = 16 columns.  What a panel does to the rows and
// columns behind it is a rank-16 update on the matrix cores: an f64 MFMA adds
// its four products as one chain of fused multiply-adds in ascending k, so an
// element sees exactly the operations, in the order, that updating it column
// by column would give.
//
// Panels are a loop and everything in it is inlined by force.  Unrolled over
// all 64 pivots the code runs once per launch, and fetching it (some 50 KB)
// took as long as running it; called as a function (the compiler's own choice)
// inverse_rows spends 6900 cycles instead of 2700, saving its registers.
// Measured: factor and inverse of a block 60000 -> 28000 cycles, a Cholesky
// step of the 2048 x 2048 CC^T 30 -> 21 us.
constexpr int PB = 16;

typedef double (*Blk)[CB + 1];

// 16 x 16 tile at (r0, c0) of T  -=  rows r0.. of A x columns: A[r][k0 + k] B(k, c)
//   TB: B(k, c) = B[c0 + c][k0 + k] (a transposed factor), else B[k0 + k][c0 + c]
template <bool TB>
__device__ __forceinline__ void tile_update(Blk T, Blk A, Blk B, int r0, int c0, int k0, bool zero) {
  const int l = threadIdx.x & 63, l16 = l & 15, l4 = l >> 4;
  double av[PB / 4], bv[PB / 4];
#pragma unroll
  for (int q = 0; q < PB / 4; ++q) {
    av[q] = -A[r0 + l16][k0 + 4 * q + l4];
    bv[q] = TB ? B[c0 + l16][k0 + 4 * q + l4] : B[k0 + 4 * q + l4][c0 + l16];
  }
  d4 acc;
#pragma unroll
  for (int v = 0; v < 4; ++v) acc[v] = zero ? 0.0 : T[r0 + l4 + 4 * v][c0 + l16];
#pragma unroll
  for (int q = 0; q < PB / 4; ++q) acc = mfma_f64(av[q], bv[q], acc);
#pragma unroll
  for (int v = 0; v < 4; ++v) T[r0 + l4 + 4 * v][c0 + l16] = acc[v];
}

// Rows of panel p of X = L^-1, all 64 columns (one wave, lane c column c):
// forward substitution, by the diagonal of L (DIV) or by its reciprocals Rs.
// Each step reads the next column of L while it uses its own; the empty asm
// statements keep the compiler from regrouping the steps into one chain of up
// to sixteen dependent operations per row.
template <bool DIV>
__device__ __forceinline__ void inverse_rows(Blk X, Blk L, const double* Rs, int p) {
  const int c = threadIdx.x & 63, r0 = PB * p, q = c / PB;
  double y[PB], dg[PB], col[2][PB];
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    y[i] = q < p ? X[r0 + i][c] : (r0 + i == c ? 1.0 : 0.0);
    dg[i] = DIV ? L[r0 + i][r0 + i] : Rs[r0 + i];
    if (i > 0) col[0][i] = L[r0 + i][r0];
  }
#pragma unroll
  for (int k = 0; k < PB; ++k) {
#pragma unroll
    for (int i = k + 2; i < PB; ++i) col[(k + 1) & 1][i] = L[r0 + i][r0 + k + 1];
    y[k] = DIV ? y[k] / dg[k] : y[k] * dg[k];
    asm volatile("" : "+v"(y[k]));
#pragma unroll
    for (int i = k + 1; i < PB; ++i) {
      y[i] = fma(-col[k & 1][i], y[k], y[i]);
      asm volatile("" : "+v"(y[i]));
    }
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) X[r0 + i][c] = y[i];
}

// What panel p of X does to the rows of the later panels: tiles (o, q), o > p
// >= q, dealt to nw waves (this one is w).  A tile's first update starts it.
__device__ __forceinline__ void inverse_update(Blk X, Blk L, int p, int w, int nw) {
  const int n = (CB / PB - 1 - p) * (p + 1);
#pragma unroll 1
  for (int t = w; t < n; t += nw) {
    const int q = t % (p + 1), o = p + 1 + t / (p + 1);
    tile_update<false>(X, L, X, PB * o, PB * q, PB * p, p == q);
  }
}

// Factor the block in C (LDS, lower part read) at global rows/cols base ..
// base + 63 (jb of them inside the matrix): L (lower) to adiag, W = L^-1 to
// w_out (row-major 64 x 64, zero above the diagonal) when need_w.  X and Rs
// (1 / L[k][k]) are LDS scratch.  info: first non-positive pivot (1-based,
// global), kept if already set.
//
// Wave 0 runs the pivots of a panel with lane r owning row r of its 16 columns
// in registers and other lanes' entries by readlane: no barrier and no LDS
// round trip inside half a panel (with the columns behind the pivot read back
// from LDS instead, a block took a sixth longer).  One wave issues an FP64
// operation every 5 to 9 cycles and its result takes 9, so a pivot (410 cycles)
// costs the chain through its root and its column updates.  Waves 1 to 3
// do what the previous panel left: its rows of W and its update of the tiles
// that the current panel does not need, then, beside the second half, its
// update of W.
__device__ __forceinline__ void factor_block(Blk C, Blk X, double* Rs, bool need_w, double* adiag, long lda, int jb,
                                             double* w_out, int* info, int base) {
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  constexpr int NP = CB / PB, H = PB / 2;
  double x[PB], v = 0.0, own = 1.0, mine = 0.0;  // own: this lane's pivot, mine: its reciprocal root
#pragma unroll 1
  for (int p = 0; p < NP; ++p) {
    const int c0 = PB * p;
    // pivot k beside the updates by column k - 1 of the columns behind k; the
    // fence keeps later broadcasts from piling up in scalar registers
    auto pivot = [&](int k) {
      if (k > 0) x[k] = fma(-v, readlane_d(v, c0 + k), x[k]);
      if (l == c0 + k) own = x[k];
      double s, rs;
      sqrt_rsqrt(readlane_d(x[k], c0 + k), s, rs);
#pragma unroll
      for (int c = k + 1; c < PB; ++c)
        if (k > 0) x[c] = fma(-v, readlane_d(v, c0 + c), x[c]);
      if (l == c0 + k) mine = rs;
      v = (l == c0 + k) ? s : x[k] * rs;
      x[k] = v;
      __builtin_amdgcn_sched_barrier(0);
    };
    if (w == 0) {
#pragma unroll
      for (int k = 0; k < PB; ++k) x[k] = C[l][c0 + k];
#pragma unroll
      for (int k = 0; k < H; ++k) pivot(k);
    } else if (w == 1) {
      if (need_w && p > 0) inverse_rows<false>(X, C, Rs, p - 1);
    } else if (p == 1) {  // tiles (I, J), J > p, of panel p - 1
      tile_update<true>(C, C, C, PB * w, PB * 2, c0 - PB, false);
      if (w == 3) tile_update<true>(C, C, C, PB * 3, PB * 3, c0 - PB, false);
    } else if (p == 2 && w == 2) {
      tile_update<true>(C, C, C, PB * 3, PB * 3, c0 - PB, false);
    }
    __syncthreads();
    if (w == 0) {
#pragma unroll
      for (int k = H; k < PB; ++k) pivot(k);
#pragma unroll
      for (int k = 0; k < PB; ++k) C[l][c0 + k] = x[k];
      if (l >= c0 && l < c0 + PB) Rs[l] = mine;
    } else if (need_w && p > 0) {
      inverse_update(X, C, p - 1, w - 1, 3);
    }
    __syncthreads();
    // panel p + 1 first: tiles (I, p + 1)
    if (w < NP - 1 - p) tile_update<true>(C, C, C, PB * (p + 1 + w), PB * (p + 1), c0, false);
    __syncthreads();
  }
  if (w == 0) {
    const unsigned long long not_pos = __ballot(!(own > 0.0));
    if (l == 0 && not_pos && *info == 0) *info = base + __ffsll((long long)not_pos);
    if (need_w) inverse_rows<false>(X, C, Rs, NP - 1);
  } else {
    for (int r = w - 1; r < CB; r += 3)
      if (r < jb && l <= r) adiag[(long)r * lda + l] = C[r][l];
  }
  __syncthreads();
  if (need_w) {
#pragma unroll
    for (int i = 0; i < CB / 4; ++i) {
      const int r = w + 4 * i;
      w_out[r * CB + l] = X[r][l];
    }
  }
}

__device__ inline void lower_tile_of(int t, int& ti, int& tj) {
  int i = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while ((i + 1) * (i + 2) / 2 <= t) ++i;
  while (i * (i + 1) / 2 > t) --i;
  ti = i;
  tj = t - i * (i + 1) / 2;
}

// Two blocks of LDS (W is read into registers): 67 KB, and at most 256
// registers, fit beside one workgroup of the ZC^T GEMM on the other stream; with
// 100 KB a step waited until a CU had none of them left.  The waves go first
// where they share a SIMD with it: a step is a chain of latencies that everything
// else waits for (half-rotated 48^3 points, K 1024: 5.60 ms without, 5.42 with).
// Alone a step of the 2048 x 2048 CC^T takes 20 us: block factor and inverse 13,
// two 64^3 products on the matrix cores 3.5, loads and launch the rest.
__global__ __launch_bounds__(CT, 2) void chol_step(double* a, long lda, int k, int nb, int j,
                                                   const double* __restrict__ w_in, double* __restrict__ w_out,
                                                   int* info) {
  __shared__ double Xi[CB][CB + 1];
  __shared__ double Xj[CB][CB + 1];
  __shared__ double Rs[CB];
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  __builtin_amdgcn_s_setprio(3);
  int ti, tj;
  lower_tile_of((int)blockIdx.x, ti, tj);
  const int I = j + 1 + ti, J = j + 1 + tj;
  const long rI = (long)I * CB, rJ = (long)J * CB;
  const bool factor = blockIdx.x == 0;  // tile (j + 1, j + 1)
  if (j >= 0) {
    const long cj = (long)j * CB;
    // wave w loads rows 16 w .. of everything, whole rows at a time
    double vi[CB / 4], vw[CB / 4], vj[CB / 4], wf[CB / 4][4];
#pragma unroll
    for (int i = 0; i < CB / 4; ++i) {
      vi[i] = ext_at(a, lda, k, rI + 16 * w + i, cj + l);
      vw[i] = w_in[(16 * w + i) * CB + l];
    }
    if (J != I) {
#pragma unroll
      for (int i = 0; i < CB / 4; ++i) vj[i] = ext_at(a, lda, k, rJ + 16 * w + i, cj + l);
    }
    d4 acc[4];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[cb][v] = ext_at(a, lda, k, rI + 16 * w + (l >> 4) + 4 * v, rJ + 16 * cb + (l & 15));
#pragma unroll
    for (int i = 0; i < CB / 4; ++i) {
      Xi[16 * w + i][l] = vi[i];
      Xj[16 * w + i][l] = vw[i];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < CB / 4; ++q)
#pragma unroll
      for (int cb = q / 4; cb < 4; ++cb) wf[q][cb] = Xj[16 * cb + (l & 15)][4 * q + (l >> 4)];
    panel_rows(Xi, wf);
    if (J != I) {
      __syncthreads();  // W has been read: its block takes A_Jj
#pragma unroll
      for (int i = 0; i < CB / 4; ++i) Xj[16 * w + i][l] = vj[i];
      panel_rows(Xj, wf);
    }
    __syncthreads();
    const double(*Lj)[CB + 1] = (J != I) ? Xj : Xi;
    if (I == J) {
      // L_I^T parked in the upper block (j, I): a[cj + c][rI + r] = L_I[r][c]
#pragma unroll
      for (int i = 0; i < CB / 4; ++i) {
        const int c = w + 4 * i;
        if (rI + l < k) a[(cj + c) * lda + rI + l] = Xi[l][c];
      }
    }
#pragma unroll
    for (int q0 = 0; q0 < CB; q0 += 4) {
      const double av = -Xi[16 * w + (l & 15)][q0 + (l >> 4)];
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) acc[cb] = mfma_f64(av, Lj[16 * cb + (l & 15)][q0 + (l >> 4)], acc[cb]);
    }
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long r = rI + 16 * w + (l >> 4) + 4 * v, c = rJ + 16 * cb + (l & 15);
        if (r < k && c < k) a[r * lda + c] = acc[cb][v];
      }
    if (!factor) return;
    // I == J here, so Xj is free; the other waves read only Xi
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
#pragma unroll
      for (int v = 0; v < 4; ++v) Xj[16 * w + (l >> 4) + 4 * v][16 * cb + (l & 15)] = acc[cb][v];
  } else {
    if (!factor) return;  // step -1 is launched as one workgroup
    load_tile(a, lda, k, 0, 0, Xj);
  }
  __syncthreads();
  factor_block(Xj, Xi, Rs, j + 2 < nb, a + rI * lda + rI, lda, (int)std::min<long>(CB, k - rI), w_out, info,
               (int)rI);
}

// Parked panels into the lower triangle, upper triangle zeroed: workgroup
// per lower block (I, p); the upper block (p, I) holds L(I, p) transposed.
__global__ __launch_bounds__(CT) void chol_finish(double* a, long lda, int k) {
  __shared__ double S[CB][CB + 1];
  int I, p;
  lower_tile_of((int)blockIdx.x, I, p);
  const int c = threadIdx.x & 63, rb = threadIdx.x >> 6;
  const long rI = (long)I * CB, rp = (long)p * CB;
  if (I == p) {
#pragma unroll
    for (int i = 0; i < CB / 4; ++i) {
      const int r = rb + 4 * i;
      if (c > r && rI + c < k) a[(rI + r) * lda + rI + c] = 0.0;
    }
    return;
  }
  const bool col_ok = rI + c < k;
  double v[CB / 4];
#pragma unroll
  for (int i = 0; i < CB / 4; ++i) v[i] = a[col_ok ? (rp + rb + 4 * i) * lda + rI + c : 0];
#pragma unroll
  for (int i = 0; i < CB / 4; ++i) {
    S[rb + 4 * i][c] = v[i];
    if (col_ok) a[(rp + rb + 4 * i) * lda + rI + c] = 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < CB / 4; ++i) {
    const int r = rb + 4 * i;
    if (rI + r < k) a[(rI + r) * lda + rp + c] = S[c][r];
  }
}

__global__ __launch_bounds__(256) void zero_upper_kernel(double* a, int k, long lda) {
  const long total = (long)k * k;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += 256L * gridDim.x) {
    const long r = e / k, c = e % k;
    if (c > r) a[r * lda + c] = 0.0;
  }
}

__global__ __launch_bounds__(256) void symmetrize_kernel(double* a, int k, long lda) {
  const long total = (long)k * k;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += 256L * gridDim.x) {
    const long r = e / k, c = e % k;
    if (c > r) a[r * lda + c] = a[c * lda + r];
  }
}

// Lp (kp x kp) = [[L, 0], [0, I]] with the strict upper part zero.
__global__ __launch_bounds__(256) void pad_lower(const double* l, int k, long lda, double* lp, int kp) {
  const long total = (long)kp * kp;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += 256L * gridDim.x) {
    const long r = e / kp, c = e % kp;
    double v = 0.0;
    if (r < k && c < k) v = (c <= r) ? l[r * lda + c] : 0.0;
    else if (r == c) v = 1.0;
    lp[e] = v;
  }
}

// Invert each 64 x 64 lower diagonal block of lp into linv (same positions),
// one block per workgroup.
__global__ __launch_bounds__(CT) void invert_diag_blocks(const double* lp, int kp, double* linv) {
  __shared__ double Ls[CB][CB + 1];
  __shared__ double Xs[CB][CB + 1];
  const long j0 = (long)blockIdx.x * CB;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  load_tile(lp, kp, kp, j0, j0, Ls);
  __syncthreads();
#pragma unroll 1
  for (int p = 0; p < CB / PB; ++p) {
    if (w == 0) inverse_rows<true>(Xs, Ls, nullptr, p);
    __syncthreads();
    inverse_update(Xs, Ls, p, w, 4);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < CB / 4; ++i) linv[(j0 + w + 4 * i) * kp + j0 + l] = Xs[w + 4 * i][l];
}

__global__ __launch_bounds__(256) void fill_zero(double* a, long count) {
  for (long e = blockIdx.x * 256L + threadIdx.x; e < count; e += 256L * gridDim.x) a[e] = 0.0;
}

inline int grid_for(long count) { return (int)std::min<long>(4096, std::max<long>(1, (count + 255) / 256)); }

// ---- symmetric tridiagonal reduction (rank of CC^T) -------------------------
// Householder reduction A = Q T Q^T of a symmetric k x k matrix, one launch
// per column j.  Launch j applies the rank-2 update of reflection j - 1
// (A22 -= v w^T + w v^T, w = p - (beta/2)(p.v) v) to the rows it owns, forms
// the updated row j in every workgroup (row j is read, never written, in this
// launch), takes reflection j from it (v = x - alpha e1, beta = 1/(alpha
// (alpha - x0)), alpha = -sign(x0) |x|), and multiplies its updated rows by v
// (p = beta A22 v).  The diagonal d and off-diagonal e of T go to d, e.
//
// A launch moves the trailing matrix once through the CUs (33 MB read and
// written at k = 2048) and is otherwise a chain of two block sums.  Each wave
// takes a whole row in registers, and its loads are issued before the chain,
// so the chain's latency hides the matrix read; row i belongs to workgroup
// i mod TD_WG in every launch, so it stays in the L2 of one XCD.  Measured at
// k = 2048: 15.9 ms for the whole rank, 7.7 us per column; with one workgroup
// of four waves per row at a time on 128 CUs, loading after the chain, it was
// 54.2 ms (45-51 us per column at full width, 1.4 TB/s).
constexpr int TD_MAXK = 4096;
constexpr int TD_WG = 256, TD_W = 8;  // workgroups (one per CU), waves of each

__device__ inline double td_block_sum(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < TD_W; ++q) s += red[q];
  return s;
}

// CH: 128-column chunks of the widest row (k <= 128 CH); the rows of W are ld
// doubles apart (a multiple of 128, zero beyond k), vp .. pn hold ld entries.
template <int CH>
__global__ __launch_bounds__(64 * TD_W) void tridiag_step(double* __restrict__ W, int ld, int k, int j,
                                                          const double* __restrict__ vp,
                                                          const double* __restrict__ pp,
                                                          const double* __restrict__ bp, double* __restrict__ vn,
                                                          double* __restrict__ pn, double* __restrict__ bn,
                                                          double* __restrict__ d, double* __restrict__ e) {
  constexpr int NT = 64 * TD_W, PT = CH * 128 / NT > 0 ? CH * 128 / NT : 1;
  __shared__ __attribute__((aligned(16))) double sv[CH * 128], sw[CH * 128], sx[CH * 128];
  __shared__ double red[2][TD_W];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const bool upd = j > 0;
  const int cb = j & ~127;  // the chunks from column j on
  const int nch = (ld - cb) >> 7, ncol = ld - cb;
  // first row > j of this wave: rows i = blockIdx + TD_WG (wave + TD_W q)
  int i = blockIdx.x + TD_WG * wave;
  if (i <= j) i += (j - i + TD_WG * TD_W) / (TD_WG * TD_W) * (TD_WG * TD_W);
  if (blockIdx.x != 0 && (int)blockIdx.x + (k - 1 - (int)blockIdx.x) / TD_WG * TD_WG <= j) return;  // no row left
  double2 x[CH];
  double2* row = reinterpret_cast<double2*>(W + (long)i * ld + cb) + lane;
  if (i < k) {
#pragma unroll
    for (int q = 0; q < CH; ++q)
      if (q < nch) x[q] = row[64 * q];
  }
  // w of reflection j - 1 and row j, columns c = cb + t + NT q
  double v[PT], w[PT], r[PT];
  double g = 0.0;
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const int c = t + NT * q;
    const bool ok = c < ncol && cb + c >= j;
    r[q] = ok ? W[(long)j * ld + cb + c] : 0.0;
    v[q] = ok && upd ? vp[cb + c] : 0.0;
    w[q] = ok && upd ? pp[cb + c] : 0.0;
    g += w[q] * v[q];
  }
  const double vj = upd ? vp[j] : 0.0, pj = upd ? pp[j] : 0.0, hb = upd ? 0.5 * bp[0] : 0.0;
  g = td_block_sum(g, red[0]) * hb;
  const double wj = pj - g * vj;
  double nrm2 = 0.0;
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    w[q] -= g * v[q];
    r[q] -= vj * w[q] + wj * v[q];
    if (cb + t + NT * q > j) nrm2 += r[q] * r[q];
  }
  // columns up to j keep v = w = x = 0: they are done
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const int c = t + NT * q;
    if (c < ncol) {
      const bool live = cb + c > j;
      sv[c] = live ? v[q] : 0.0;
      sw[c] = live ? w[q] : 0.0;
      sx[c] = live ? r[q] : 0.0;
      if (blockIdx.x == 0 && cb + c == j) d[j] = r[q];
    }
  }
  nrm2 = td_block_sum(nrm2, red[1]);
  double alpha = 0.0, beta = 0.0;
  if (j + 1 < k && nrm2 > 0.0) {
    const double x0 = sx[j + 1 - cb];
    alpha = x0 >= 0.0 ? -sqrt(nrm2) : sqrt(nrm2);
    beta = 1.0 / (alpha * (alpha - x0));
  }
  __syncthreads();
  if (t == 0 && j + 1 < k) sx[j + 1 - cb] -= alpha;  // v = x - alpha e1
  __syncthreads();
  if (blockIdx.x == 0) {
    if (t == 0) {
      if (j + 1 < k) e[j] = alpha;
      bn[0] = beta;
    }
    for (int c = t; c < ncol; c += NT) vn[cb + c] = sx[c];
  }
  const double2* v2 = reinterpret_cast<const double2*>(sv) + lane;
  const double2* w2 = reinterpret_cast<const double2*>(sw) + lane;
  const double2* x2 = reinterpret_cast<const double2*>(sx) + lane;
  while (i < k) {
    const double vi = sv[i - cb], wi = sw[i - cb];
    double acc = 0.0;
#pragma unroll
    for (int q = 0; q < CH; ++q)
      if (q < nch) {
        const double2 a = w2[64 * q], b = v2[64 * q], c = x2[64 * q];
        x[q].x -= vi * a.x + wi * b.x;
        x[q].y -= vi * a.y + wi * b.y;
        if (upd) row[64 * q] = x[q];
        acc += x[q].x * c.x + x[q].y * c.y;
      }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) pn[i] = beta * acc;
    i += TD_WG * TD_W;
    if (i < k) {
      row = reinterpret_cast<double2*>(W + (long)i * ld + cb) + lane;
#pragma unroll
      for (int q = 0; q < CH; ++q)
        if (q < nch) x[q] = row[64 * q];
    }
  }
}

// a (k x k) into rows of ld doubles, zero beyond column k; the step vectors zeroed
__global__ __launch_bounds__(256) void copy_square(const double* a, long lda, int k, double* w, int ld, double* vec,
                                                   int nvec) {
  const long total = (long)k * ld;
  for (long q = blockIdx.x * 256L + threadIdx.x; q < total; q += 256L * gridDim.x) {
    const long r = q / ld, c = q - r * ld;
    w[q] = c < k ? a[r * lda + c] : 0.0;
  }
  for (long q = blockIdx.x * 256L + threadIdx.x; q < nvec; q += 256L * gridDim.x) vec[q] = 0.0;
}

// number of eigenvalues of the tridiagonal (d, e) below x (Sturm count of the
// LDL^T pivots of T - x I)
int sturm_count(const double* d, const double* e, int k, double x) {
  int neg = 0;
  double q = 1.0;
  for (int i = 0; i < k; ++i) {
    const double off = i > 0 ? e[i - 1] * e[i - 1] : 0.0;
    q = d[i] - x - (i > 0 ? off / q : 0.0);
    if (q == 0.0) q = -1e-300;  // an exact zero pivot counts as negative
    if (q < 0.0) ++neg;
  }
  return neg;
}

// eigenvalue of rank 'idx' (0 = smallest) by bisection within the Gershgorin
// interval, to the resolution of double
double tridiag_eig(const double* d, const double* e, int k, int idx) {
  double lo = 0.0, hi = 0.0;
  for (int i = 0; i < k; ++i) {
    const double r = (i > 0 ? std::fabs(e[i - 1]) : 0.0) + (i + 1 < k ? std::fabs(e[i]) : 0.0);
    lo = i == 0 ? d[i] - r : std::min(lo, d[i] - r);
    hi = i == 0 ? d[i] + r : std::max(hi, d[i] + r);
  }
  for (int it = 0; it < 200; ++it) {
    const double mid = 0.5 * (lo + hi);
    if (mid <= lo || mid >= hi) break;
    if (sturm_count(d, e, k, mid) > idx) hi = mid;
    else lo = mid;
  }
  return 0.5 * (lo + hi);
}

}  // namespace

size_t chol_work_bytes(int) { return 2 * align_up(sizeof(double) * CB * CB, 256); }

int cholesky_f64(double* a, int k, long lda, int* d_info, void* work, hipStream_t s) {
  if (k < 1) return THC_OK;
  // W_j lives in wb[j & 1]: step j - 1 writes it, step j reads it
  double* wb[2] = {reinterpret_cast<double*>(work),
                   reinterpret_cast<double*>(reinterpret_cast<char*>(work) + align_up(sizeof(double) * CB * CB, 256))};
  const int nb = ceil_div(k, CB);
  for (int j = -1; j < nb - 1; ++j) {
    const long tb = j < 0 ? 1 : nb - j - 1;  // step -1 has only the factor of block 0
    hipLaunchKernelGGL(chol_step, dim3((unsigned)(tb * (tb + 1) / 2)), dim3(CT), 0, s, a, lda, k, nb, j,
                       wb[(j + 2) & 1], wb[(j + 1) & 1], d_info);
    THC_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(chol_finish, dim3((unsigned)((long)nb * (nb + 1) / 2)), dim3(CT), 0, s, a, lda, k);
  THC_HIP(hipGetLastError());
  return THC_OK;
}

static int padded(int k) {
  int kp = NB;
  while (kp < k) kp *= 2;
  return kp;
}

size_t spd_inverse_work_bytes(int k) {
  const size_t kp = padded(k);
  return 3 * align_up(sizeof(double) * kp * kp, 256) + 1024;
}

int spd_inverse_from_chol(const double* l, int k, long lda, double* ainv, void* work, hipStream_t s) {
  const int kp = padded(k);
  const size_t mat = align_up(sizeof(double) * (size_t)kp * kp, 256);
  double* lp = reinterpret_cast<double*>(work);
  double* linv = reinterpret_cast<double*>(reinterpret_cast<char*>(work) + mat);
  double* tmp = reinterpret_cast<double*>(reinterpret_cast<char*>(work) + 2 * mat);
  const long kk = (long)kp * kp;
  hipLaunchKernelGGL(pad_lower, dim3(grid_for(kk)), dim3(256), 0, s, l, k, lda, lp, kp);
  hipLaunchKernelGGL(fill_zero, dim3(grid_for(kk)), dim3(256), 0, s, linv, kk);
  hipLaunchKernelGGL(invert_diag_blocks, dim3(kp / NB), dim3(CT), 0, s, lp, kp, linv);
  THC_HIP(hipGetLastError());
  for (int sz = NB; sz < kp; sz *= 2) {
    const int pairs = kp / (2 * sz);
    const long step = (long)2 * sz * kp + 2 * sz;  // diagonal stride between pairs
    // tmp_p = L21 Linv11
    GemmArgs g = {};
    g.m = sz; g.n = sz; g.k = sz;
    g.a = lp + (long)sz * kp; g.lda = kp; g.a_trans = 0;
    g.b = linv; g.ldb = kp; g.b_trans = 0;
    g.c = tmp; g.ldc = sz;
    g.alpha = 1.0; g.beta = 0.0; g.batch = pairs;
    g.tri = GEMM_TRI_B_KGE_N;  // Linv11 is lower triangular
    g.stride_a = step; g.stride_b = step; g.stride_c = (long)sz * sz;
    THC_TRY(gemm_f64(g, s));
    // Linv21 = -Linv22 tmp_p
    GemmArgs h = {};
    h.m = sz; h.n = sz; h.k = sz;
    h.a = linv + (long)sz * kp + sz; h.lda = kp; h.a_trans = 0;
    h.b = tmp; h.ldb = sz; h.b_trans = 0;
    h.c = linv + (long)sz * kp; h.ldc = kp;
    h.alpha = -1.0; h.beta = 0.0; h.batch = pairs;
    h.tri = GEMM_TRI_A_KLE_M;  // Linv22 is lower triangular
    h.stride_a = step; h.stride_b = (long)sz * sz; h.stride_c = step;
    THC_TRY(gemm_f64(h, s));
  }
  // A^-1 = Linv^T Linv (top-left k x k): lower tiles only, each over the k
  // range where both triangular operands are nonzero, then mirrored
  GemmArgs f = {};
  f.m = k; f.n = k; f.k = k;
  f.a = linv; f.lda = kp; f.a_trans = 1;
  f.b = linv; f.ldb = kp; f.b_trans = 0;
  f.c = ainv; f.ldc = k;
  f.alpha = 1.0; f.beta = 0.0; f.batch = 1;
  f.lower = 1;
  f.tri = GEMM_TRI_A_KGE_M | GEMM_TRI_B_KGE_N;
  THC_TRY(gemm_f64(f, s));
  hipLaunchKernelGGL(symmetrize_kernel, dim3(grid_for((long)k * k)), dim3(256), 0, s, ainv, k, (long)k);
  THC_HIP(hipGetLastError());
  return THC_OK;
}

inline int td_ld(int k) { return (k + 127) / 128 * 128; }

size_t tridiag_work_bytes(int k) {
  return align_up(sizeof(double) * (size_t)k * td_ld(k), 256) + 6 * align_up(sizeof(double) * (size_t)td_ld(k), 256) +
         2 * align_up(sizeof(double) * 4, 256) + 256;
}

int sym_tridiag(const double* a, int k, long lda, double* d_host, double* e_host, void* work, hipStream_t s) {
  if (k < 1) return THC_OK;
  if (k > TD_MAXK) return THC_ERR_UNSUPPORTED;
  char* w = reinterpret_cast<char*>(work);
  auto take = [&](size_t count) {
    double* p = reinterpret_cast<double*>(w);
    w += align_up(sizeof(double) * count, 256);
    return p;
  };
  const int ld = td_ld(k);
  double* W = take((size_t)k * ld);
  double* vec = take((size_t)4 * ld);  // v and p of the two latest reflections
  double* vb[2] = {vec, vec + ld};
  double* pb[2] = {vec + 2 * ld, vec + 3 * ld};
  double* bb[2] = {take(4), take(4)};
  double* dd = take(ld);
  double* ee = take(ld);
  hipLaunchKernelGGL(copy_square, dim3(grid_for((long)k * ld)), dim3(256), 0, s, a, lda, k, W, ld, vec, 4 * ld);
  THC_HIP(hipGetLastError());
  for (int j = 0; j < k; ++j) {
    const int cur = j & 1, prev = cur ^ 1;
    const int left = (ld - (j & ~127)) >> 7;  // chunks this step touches: the registers and LDS of the step follow
    auto step = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(std::min(TD_WG, k)), dim3(64 * TD_W), 0, s, W, ld, k, j, vb[prev], pb[prev],
                         bb[prev], vb[cur], pb[cur], bb[cur], dd, ee);
    };
    if (left <= 4) step(tridiag_step<4>);
    else if (left <= 8) step(tridiag_step<8>);
    else if (left <= 16) step(tridiag_step<16>);
    else step(tridiag_step<32>);
    THC_HIP(hipGetLastError());
  }
  THC_HIP(hipMemcpyAsync(d_host, dd, sizeof(double) * k, hipMemcpyDeviceToHost, s));
  if (k > 1) THC_HIP(hipMemcpyAsync(e_host, ee, sizeof(double) * (k - 1), hipMemcpyDeviceToHost, s));
  return THC_OK;
}

void tridiag_rank(const double* d, const double* e, int k, int* rank, double* smax) {
  if (k < 1) {
    *rank = 0;
    *smax = 0.0;
    return;
  }
  // singular values of a symmetric matrix are |eigenvalues|; the largest is
  // the larger magnitude of the two extreme eigenvalues
  const double lmin = tridiag_eig(d, e, k, 0), lmax = tridiag_eig(d, e, k, k - 1);
  const double s0 = std::max(std::fabs(lmin), std::fabs(lmax));
  // MatrixOperations::rank: sigma_i < max(m, n) s0 1e-16 counts as zero
  const double rcond = (double)k * s0 * 1e-16;
  const int nul = sturm_count(d, e, k, rcond) - sturm_count(d, e, k, -rcond);
  *rank = k - nul;
  *smax = s0;
}

int zero_upper(double* a, int k, long lda, hipStream_t s) {
  hipLaunchKernelGGL(zero_upper_kernel, dim3(grid_for((long)k * k)), dim3(256), 0, s, a, k, lda);
  THC_HIP(hipGetLastError());
  return THC_OK;
}

int symmetrize_from_lower(double* a, int k, long lda, hipStream_t s) {
  hipLaunchKernelGGL(symmetrize_kernel, dim3(grid_for((long)k * k)), dim3(256), 0, s, a, k, lda);
  THC_HIP(hipGetLastError());
  return THC_OK;
}

}  // namespace thc

// ---------------------------------------------------------------- no-allocation Cholesky
//
// thc_cholesky_noalloc's scratch: the two panel-inverse buffers cholesky_f64
// works in, then its info word.  A file-scope device array: each GPU the
// library runs on holds one copy, for the life of the process.  In host code
// the name 'scratch' is a host-side stand-in, never a device address; the
// device address of each GPU's copy comes from hipGetSymbolAddress, taken once
// per device (from thc_ctx_create, with that device current) and kept below.
namespace thc {
namespace {
constexpr size_t kCholScratchWork = 2 * 64 * 64 * sizeof(double);  // chol_work_bytes(): two 64 x 64 panels
constexpr size_t kCholScratchBytes = kCholScratchWork + 256;        // + the info word (256-byte slot)
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace
}  // namespace thc

static __device__ __attribute__((aligned(256))) unsigned char scratch[thc::kCholScratchBytes];

namespace thc {

int noalloc_scratch_init(int device) {
  if (device < 0 || device >= kMaxDevices) return THC_ERR_UNSUPPORTED;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return THC_OK;
  void* p = nullptr;
  THC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = p;
  return THC_OK;
}

namespace {
__global__ void zero_info(int* p) {
  if (threadIdx.x == 0) *p = 0;
}
}  // namespace

}  // namespace thc

extern "C" int thc_cholesky_noalloc(thc_ctx* ctx, double* a, int k, int* info) {
  using namespace thc;
  if (!ctx || !a || !info || k < 1) return THC_ERR_ARG;
  if (chol_work_bytes(k) > kCholScratchWork) {
    set_last_error("thc_cholesky_noalloc: the Cholesky panels need more than the static scratch holds", __FILE__,
                   __LINE__);
    return THC_ERR_UNSUPPORTED;
  }
  if (ctx->device < 0 || ctx->device >= kMaxDevices) return THC_ERR_UNSUPPORTED;
  if (!ctx->pinned || ctx->pinned_bytes < sizeof(int)) return THC_ERR_ARG;  // thc_ctx_create provides it
  THC_HIP(hipSetDevice(ctx->device));
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    base = g_scratch_ptr[ctx->device];
  }
  if (!base) THC_TRY(noalloc_scratch_init(ctx->device));  // a device the library was not set up on
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    base = g_scratch_ptr[ctx->device];
  }
  double* work = reinterpret_cast<double*>(base);
  int* d_info = reinterpret_cast<int*>(reinterpret_cast<char*>(base) + kCholScratchWork);
  hipLaunchKernelGGL(zero_info, dim3(1), dim3(64), 0, ctx->stream, d_info);
  THC_HIP(hipGetLastError());
  THC_TRY(cholesky_f64(a, k, k, d_info, work, ctx->stream));
  int* h = reinterpret_cast<int*>(ctx->pinned);
  THC_HIP(hipMemcpyAsync(h, d_info, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  THC_HIP(hipStreamSynchronize(ctx->stream));
  *info = *h;
  return THC_OK;
}
