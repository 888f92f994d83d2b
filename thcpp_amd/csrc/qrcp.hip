// Interpolation points by QR with column pivoting (QRCPSolver::kernel,
// src/qrcp.cpp:100-173; pzgeqpf at src/matrix_operations.h:756-788) without
// forming the orbital-product matrix.
//
// The reference factors ZT[(i k), a] = phi_i(r_a) phi_k(r_a) (M^2 x N; for the
// half-rotated set, i runs over the occupied orbitals) and keeps the first K
// pivot columns.  Column pivoting only ever looks at inner products of
// columns, and those are
//   <Z_a, Z_b> = (sum_i phi_i(a) phi_i(b)) (sum_k phi_k(a) phi_k(b)),
// i.e. the Gram matrix G = P o Pocc (P o P without half rotation).  Pivoted
// Cholesky of G picks, step by step, the column of largest residual norm and
// projects it out -- the same pivots as QR with column pivoting of ZT in exact
// arithmetic, with the pivot's residual norm equal to |R_jj|.  A step is
//   p      = argmax residual d (first index on ties);
//   g_a    = G[a][p] from two M-length dot products with the pivot's row;
//   l_a    = (g_a - sum_{q<j} L[q][a] L[q][p]) / sqrt(d_p);
//   d_a   -= l_a^2  (the pivot itself is retired),
// and reads all j earlier columns of L, N j doubles, for one column.  Residuals
// only ever fall, so several steps can share that read: take as candidates all
// points with residual above some bound (at most QC of them).  As long as the
// largest candidate residual stays above the bound, no other point can be the
// next pivot, and the steps run on the candidates' own QC x QC block of the
// Schur complement.  A round (real G) is
//   qr_pick    candidates: all points in the top bins of a histogram of d;
//   qr_gather  their columns of L, qr_gram their block G - L L^T (MFMA);
//   qr_run     the pivot steps on that block, up to QR_MAX of them;
//   qr_apply   the chosen columns for all N points at once: one pass over L
//              (MFMA), a triangular solve, the new d, its histogram and maxima.
// On a 40^3 grid, M = 64, K = 512: 27 rounds of 19 pivots on average, 2.8 ms
// (qr_apply 44 us, qr_run 28 us a round); one kernel per pivot, each reading
// all earlier columns, took 17.7 ms (8 us + 0.085 us per earlier column).
// QC = 256 candidates: 128 give 37 rounds, 512 give 21 with a four times
// larger block.
//
// Where more than QC points share the top bin -- symmetry-equivalent points of a
// crystal, whose residuals are equal -- no set of candidates holds every point
// that may be next.  The run then goes on one pivot a step (qr_step), and tries
// a round again after 4, 8, ... 32 of them.
//
// Complex orbitals (ZT[(i k), a] = conj(phi_i(r_a)) phi_k(r_a), src/qrcp.cpp:
// 33-48): with Q[a][b] = sum_k conj(phi_k(a)) phi_k(b) the Gram matrix is
// conj(Q) o Q = |Q|^2, real, and the steps above apply with g_a = |Q[a][p]|^2.
// Half-rotated (i over the occupied set) it is conj(Qocc) o Q, Hermitian: the
// columns of L are complex, l_a = (G[a][p] - sum_q L[a][q] conj(L[p][q])) /
// sqrt(d_p) and d_a -= |l_a|^2; the residual norms, hence the pivots, are
// those of QR with column pivoting of the complex ZT.
#include <algorithm>
#include <cfloat>
#include <type_traits>
#include <vector>

#include "common.h"

namespace thc {
namespace {

constexpr int QB = 256;          // threads per block
constexpr double RETIRED = -DBL_MAX;  // residual of a chosen point (no arithmetic reaches it)

__device__ inline bool wins(double v, int i, double bv, int bi) { return v > bv || (v == bv && i < bi); }

// (max value, first index) over the block into pv/pi[blockIdx.x]
__device__ void block_argmax(double v, int i, double* pv, int* pi) {
  __shared__ double sv[QB / 64];
  __shared__ int si[QB / 64];
  for (int o = 32; o > 0; o >>= 1) {
    const double ov = __shfl_xor(v, o);
    const int oi = __shfl_xor(i, o);
    if (wins(ov, oi, v, i)) { v = ov; i = oi; }
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { sv[w] = v; si[w] = i; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < QB / 64; ++q)
      if (wins(sv[q], si[q], v, i)) { v = sv[q]; i = si[q]; }
    pv[blockIdx.x] = v;
    pi[blockIdx.x] = i;
  }
}

__device__ inline double dot_row(const double* __restrict__ x, const double* __restrict__ y, int m) {
  double s0 = 0.0, s1 = 0.0;
  int q = 0;
  for (; q + 2 <= m; q += 2) {
    s0 = fma(x[q], y[q], s0);
    s1 = fma(x[q + 1], y[q + 1], s1);
  }
  if (q < m) s0 = fma(x[q], y[q], s0);
  return s0 + s1;
}

// sum_q conj(x_q) y_q over interleaved complex rows (m2 doubles)
__device__ inline void cdot_row(const double* __restrict__ x, const double* __restrict__ y, int m2, double& re,
                                double& im) {
  double r = 0.0, i = 0.0;
  for (int q = 0; q + 2 <= m2; q += 2) {
    r = fma(x[q], y[q], r);
    r = fma(x[q + 1], y[q + 1], r);
    i = fma(x[q], y[q + 1], i);
    i = fma(-x[q + 1], y[q], i);
  }
  re = r;
  im = i;
}

// d_a = G[a][a] and the first per-block maxima (sum |phi|^2 over interleaved
// complex rows is the real row's dot product, so one kernel serves both)
__global__ __launch_bounds__(QB) void qr_init(const double* __restrict__ phi, const double* __restrict__ occ, long n,
                                              int m, int mo, double* __restrict__ d, double* pv, int* pi) {
  const long a = (long)blockIdx.x * QB + threadIdx.x;
  double v = -DBL_MAX;
  int vi = INT_MAX;
  if (a < n) {
    const double* x = phi + a * m;
    const double s = dot_row(x, x, m);
    double g = s * s;
    if (occ) {
      const double* y = occ + a * mo;
      g = s * dot_row(y, y, mo);
    }
    d[a] = g;
    v = g;
    vi = (int)a;
  }
  block_argmax(v, vi, pv, pi);
}

// ---- rounds of pivots for a real G --------------------------------------------

constexpr int QC = 256;       // candidates of a round (threads of qr_run)
constexpr int QR_MAX = 32;    // pivots of a round: two MFMA tiles of columns
constexpr int QBINS = 1536;   // bins of the residual histogram: 128 an octave, 12 octaves below the reference
constexpr int QBIN_SHIFT = 13;  // a residual's bin: the exponent and 7 mantissa bits of its high word

// G = P^2, P Pocc, |P|^2 (complex), conj(Pocc) P (complex half-rotated: G itself is complex)
enum { G_SQUARE = 0, G_PRODUCT = 1, G_MODULUS = 2, G_COMPLEX = 3 };

struct QrState {
  int j, done, stall;  // pivots chosen, run ended, no candidates to be had: read back together
  int base, r;      // pivots chosen before this round, chosen in it
  int ncand, cut;   // candidates, the lowest bin (counted downwards) that is among them
  int refkey;       // bin key no residual is above
  int slot[QR_MAX];  // candidate slots of the round's pivots
  int piv[QR_MAX];
  double rs[QR_MAX];            // 1 / sqrt(residual) of the pivots
  double tri[QR_MAX][QR_MAX];   // tri[s][t] = l_s at pivot t > s
};

__device__ inline int qr_key(double v) { return (int)(__double_as_longlong(v) >> 32) >> QBIN_SHIFT; }
// bin of a positive residual, counted downwards from the reference; QBINS and
// above are out of range
__device__ inline int qr_bin(double v, int refkey) { return max(0, refkey - qr_key(v)); }

// first maximum over nparts per-block maxima, to all threads of the block
__device__ inline void qr_top(const double* pv, const int* pi, int nparts, double& v, int& vi, double* sv, int* si) {
  v = -DBL_MAX;
  vi = INT_MAX;
  for (int q = threadIdx.x; q < nparts; q += blockDim.x)
    if (wins(pv[q], pi[q], v, vi)) { v = pv[q]; vi = pi[q]; }
  for (int o = 32; o > 0; o >>= 1) {
    const double ov = __shfl_xor(v, o);
    const int oi = __shfl_xor(vi, o);
    if (wins(ov, oi, v, vi)) { v = ov; vi = oi; }
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) { sv[w] = v; si[w] = vi; }
  __syncthreads();
  v = sv[0];
  vi = si[0];
  for (int q = 1; q < (int)(blockDim.x >> 6); ++q)
    if (wins(sv[q], si[q], v, vi)) { v = sv[q]; vi = si[q]; }
}

// Start of the rounds with j of k pivots chosen: the reference residual, an
// empty histogram.
__global__ __launch_bounds__(QB) void qr_begin(const double* pv, const int* pi, int nparts, int j, int k, int* fail,
                                               QrState* st, int* hist) {
  __shared__ double sv[QB / 64];
  __shared__ int si[QB / 64];
  double v;
  int vi;
  qr_top(pv, pi, nparts, v, vi, sv, si);
  if (threadIdx.x == 0) {
    st->j = j;
    st->base = st->r = st->ncand = st->stall = 0;
    if (j == 0) *fail = 0;
    st->done = *fail || j >= k;
    st->cut = -1;
    st->refkey = v > 0.0 ? qr_key(v) : 0;
  }
  for (int b = threadIdx.x; b < QBINS; b += QB) hist[b] = 0;
}

// The block's residuals (one a thread) into the histogram, through LDS.
__device__ inline void qr_count(double v, int refkey, int* h, int* hist) {
  for (int b = threadIdx.x; b < QBINS; b += blockDim.x) h[b] = 0;
  __syncthreads();
  if (v > 0.0) {
    const int b = qr_bin(v, refkey);
    if (b < QBINS) atomicAdd(&h[b], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < QBINS; b += blockDim.x)
    if (h[b]) atomicAdd(&hist[b], h[b]);
}

__global__ __launch_bounds__(QB) void qr_hist(const double* __restrict__ d, long n, const QrState* st, int* hist) {
  __shared__ int h[QBINS];
  const long a = (long)blockIdx.x * QB + threadIdx.x;
  qr_count(a < n ? d[a] : 0.0, st->refkey, h, hist);
}

// Candidates: the points of the most bins from the top that hold at most QC
// of them.  None if the top bin alone holds more (or nothing is in range).
__global__ __launch_bounds__(QB) void qr_pick(const double* __restrict__ d, long n, const int* __restrict__ hist,
                                              QrState* st, int* cand) {
  if (st->done || st->stall) return;
  constexpr int PER = QBINS / QB;
  static_assert(PER * QB == QBINS, "bins split evenly over the threads");
  __shared__ int part[QB];
  __shared__ int cut;
  const int t = threadIdx.x;
  const int refkey = st->refkey;
  int c[PER], sum = 0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    c[q] = hist[t * PER + q];
    sum += c[q];
  }
  part[t] = sum;
  if (t == 0) cut = -1;
  __syncthreads();
  for (int o = 1; o < QB; o <<= 1) {
    const int v = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int run = part[t] - sum;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    run += c[q];
    if (run > 0 && run <= QC) atomicMax(&cut, t * PER + q);
  }
  __syncthreads();
  if (blockIdx.x == 0 && t == 0) st->cut = cut;
  if (cut < 0) return;
  const long a = (long)blockIdx.x * QB + t;
  const double v = a < n ? d[a] : 0.0;
  if (v > 0.0 && qr_bin(v, refkey) <= cut) cand[atomicAdd(&st->ncand, 1)] = (int)a;
}

// LT[q][t] = L[q][cand[t]], q < j, zero for rows up to the next multiple of 4
// and slots without a candidate.
__global__ __launch_bounds__(QC) void qr_gather(const double* __restrict__ L, long ln, const QrState* st,
                                                const int* __restrict__ cand, double* __restrict__ LT) {
  if (st->done || st->ncand == 0) return;
  const int t = threadIdx.x, j = st->j, j4 = (j + 3) & ~3;
  const bool ok = t < st->ncand;
  const double* src = L + (ok ? cand[t] : 0);
  for (int q = blockIdx.x; q < j4; q += gridDim.x) LT[(long)q * QC + t] = ok && q < j ? src[q * ln] : 0.0;
}

typedef double qd4 __attribute__((ext_vector_type(4)));
__device__ inline qd4 qr_mfma(double a, double b, qd4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// entry k of i phi at point p (interleaved): against phi it gives the imaginary part of P
__device__ inline double qr_times_i(const double* __restrict__ phi, long p, int m, int k) {
  const double v = phi[p * m + (k ^ 1)];
  return k & 1 ? -v : v;
}
template <int G>
__device__ inline double qr_combine(double p, double q) {
  return G == G_SQUARE ? p * p : (G == G_PRODUCT ? p * q : p * p + q * q);
}

// S = G - L L^T over the candidates: one 16 x 16 tile per workgroup, the inner
// dimensions split over its four waves.
template <int G>
__global__ __launch_bounds__(256) void qr_gram(const double* __restrict__ phi, const double* __restrict__ occ, int m,
                                               int mo, const QrState* st, const int* __restrict__ cand,
                                               const double* __restrict__ LT, double* __restrict__ S) {
  const int nc = st->ncand;
  const int I = (blockIdx.x & 15) * 16, J = (blockIdx.x >> 4) * 16;
  if (st->done || I >= nc || J >= nc) return;
  __shared__ double red[3][4][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l16 = lane & 15, l4 = lane >> 4;
  const int j4 = (st->j + 3) >> 2;
  qd4 acc = {}, p1 = {}, p2 = {};
  {
    const int per = (j4 + 3) / 4, q0 = w * per, q1 = min(j4, q0 + per);
    const double* base = LT + (long)l4 * QC + l16;
    for (int q = q0; q < q1; q += 8) {  // eight steps' loads in flight
      double x[8], y[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const double* row = base + (long)min(q + u, q1 - 1) * 4 * QC;
        x[u] = row[I];
        y[u] = row[J];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (q + u < q1) acc = qr_mfma(x[u], y[u], acc);
    }
  }
  const long pi = I + l16 < nc ? cand[I + l16] : cand[0], pj = J + l16 < nc ? cand[J + l16] : cand[0];
  for (int k0 = 4 * w; k0 < m; k0 += 64) {
    double x[4], y[4], z[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = k0 + 16 * u + l4;
      const bool ok = k < m;
      x[u] = ok ? phi[pi * m + k] : 0.0;
      y[u] = ok ? phi[pj * m + k] : 0.0;
      z[u] = G == G_MODULUS && ok ? qr_times_i(phi, pj, m, k) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      p1 = qr_mfma(x[u], y[u], p1);
      if (G == G_MODULUS) p2 = qr_mfma(x[u], z[u], p2);
    }
  }
  if (G == G_PRODUCT)
    for (int k0 = 4 * w; k0 < mo; k0 += 64) {
      double x[4], y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + 16 * u + l4;
        x[u] = k < mo ? occ[pi * mo + k] : 0.0;
        y[u] = k < mo ? occ[pj * mo + k] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) p2 = qr_mfma(x[u], y[u], p2);
    }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int o = (l4 + 4 * v) * 16 + l16;
    red[0][w][o] = acc[v];
    red[1][w][o] = p1[v];
    if (G != G_SQUARE) red[2][w][o] = p2[v];
  }
  __syncthreads();
  const int t = threadIdx.x;
  double sum[3] = {};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    sum[0] += red[0][q][t];
    sum[1] += red[1][q][t];
    if (G != G_SQUARE) sum[2] += red[2][q][t];
  }
  S[(long)(I + (t >> 4)) * QC + J + (t & 15)] = qr_combine<G>(sum[1], sum[2]) - sum[0];
}

// v, or where the DPP control moves a lane's value there, the larger of the two
template <int CTRL, int ROWS>
__device__ inline double qr_dpp_max(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return fmax(v, __longlong_as_double(((long long)hi << 32) | (unsigned)lo));
}
// maximum over the wave: within rows of 16 by shifts, then lane 15 of a row to
// the next and lane 31 to the upper half; lane 63 holds it
__device__ inline double qr_wave_max(double v) {
  v = qr_dpp_max<0x111, 0xf>(v);
  v = qr_dpp_max<0x112, 0xf>(v);
  v = qr_dpp_max<0x114, 0xf>(v);
  v = qr_dpp_max<0x118, 0xf>(v);
  v = qr_dpp_max<0x142, 0xa>(v);
  v = qr_dpp_max<0x143, 0xc>(v);
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Pivot steps on the candidates, until the largest residual falls out of
// their bins.  The first pivot of a round is the first maximum over all points
// in any case: the candidates hold every point of the top bin; without
// candidates the round ends here (stall).  One wave, four
// candidates a lane (lane l owns l, l + 64, ...), so a step is a chain without
// barriers: the maximum over the lanes, one row of S, r multiply-adds.  The
// other waves read S once, so that its rows are in this XCD's L2 by then.
__global__ __launch_bounds__(1024) void qr_run(const double* __restrict__ S, const double* __restrict__ d,
                                             const int* __restrict__ cand, int k, QrState* st, int* __restrict__ hist,
                                             int* __restrict__ piv, double* __restrict__ rdiag,
                                             int* __restrict__ fail_out) {
  if (st->done || st->stall) return;
  constexpr int PL = QC / 64;
  __shared__ double lh[QR_MAX][QC];
  const int lane = threadIdx.x & 63;
  const int j = st->j, nc = st->ncand, cut = st->cut, refkey = st->refkey;
  if (threadIdx.x >= 64) {
    double sum = 0.0;
    const int lines = (nc + 15) / 16;  // 128-byte lines of a row's first nc entries
    for (int q = threadIdx.x - 64; q < nc * lines; q += 1024 - 64) sum += S[(long)(q / lines) * QC + q % lines * 16];
    asm volatile("" ::"v"(sum));
    return;
  }
  if (cut < 0) {
    if (lane == 0) st->stall = 1;
    return;
  }
  int me[PL];
  double dt[PL];
#pragma unroll
  for (int u = 0; u < PL; ++u) {
    const int t = lane + 64 * u;
    me[u] = t < nc ? cand[t] : INT_MAX;
    dt[u] = t < nc ? d[me[u]] : -DBL_MAX;
  }
  double d0 = j > 0 ? rdiag[0] * rdiag[0] : 0.0;
  int newkey = refkey, fail = 0, r = 0;
  for (; r < QR_MAX && j + r < k; ++r) {
    double v = dt[0];
    int vi = me[0], vs = lane;
#pragma unroll
    for (int u = 1; u < PL; ++u)
      if (wins(dt[u], me[u], v, vi)) { v = dt[u]; vi = me[u]; vs = lane + 64 * u; }
    const double top = qr_wave_max(v);
    unsigned long long at = __ballot(v == top);
    if (__popcll(at) > 1) {  // equal residuals: the first point
      int low = v == top ? vi : INT_MAX;
      for (int o = 32; o > 0; o >>= 1) low = min(low, __shfl_xor(low, o));
      at = __ballot(v == top && vi == low);
    }
    const int win = at ? __ffsll((long long)at) - 1 : 0;
    v = top;
    vi = __builtin_amdgcn_readlane(vi, win);
    vs = __builtin_amdgcn_readlane(vs, win);
    if (r > 0 && (!(v > 0.0) || qr_bin(v, refkey) > cut)) break;
    if (j + r == 0) d0 = v;
    // residual exhausted (K beyond the numerical rank): below 1e-13 of the first
    // pivot the squared residuals are rounding noise of the Gram downdate
    if (nc == 0 || !(v > 1e-13 * d0)) { fail = j + r + 1; break; }
    if (r == 0) newkey = qr_key(v);
    double c[PL];
#pragma unroll
    for (int u = 0; u < PL; ++u) c[u] = lane + 64 * u < nc ? S[(long)vs * QC + lane + 64 * u] : 0.0;
    const double rt = sqrt(v), rs = 1.0 / rt;
    const double mine = lane < r ? lh[lane & (QR_MAX - 1)][vs] : 0.0;
#pragma unroll 4
    for (int q = 0; q < r; ++q) {
      const double f = lh[q][vs];
#pragma unroll
      for (int u = 0; u < PL; ++u) c[u] -= lh[q][lane + 64 * u] * f;
    }
#pragma unroll
    for (int u = 0; u < PL; ++u) {
      const double l = c[u] * rs;
      lh[r][lane + 64 * u] = l;
      if (lane + 64 * u == vs) dt[u] = RETIRED;
      else if (dt[u] != RETIRED) dt[u] -= l * l;
    }
    if (lane == 0) {
      st->slot[r] = vs;
      st->piv[r] = vi;
      st->rs[r] = rs;
      piv[j + r] = vi;
      rdiag[j + r] = rt;
    }
    if (lane < r) st->tri[lane][r] = mine;
    // the next step's reads of lh follow these writes in the wave's own order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
  for (int b = lane; b < QBINS; b += 64) hist[b] = 0;
  if (lane == 0) {
    st->base = j;
    st->r = r;
    st->j = j + r;
    st->ncand = 0;
    st->refkey = newkey;
    if (fail) *fail_out = fail;  // the step that found no pivot, 1-based
    st->done = fail || j + r >= k;
  }
}

// The pivots' columns of LT side by side, LP[q][s] (zero for s >= r), so that
// qr_apply reads them in whole lines: with every wave gathering them from LT
// the 40^3, K = 512 run took 3.05 ms, with this kernel 2.80.
__global__ __launch_bounds__(256) void qr_compact(const QrState* st, const double* __restrict__ LT,
                                                  double* __restrict__ LP) {
  if (st->done || st->stall) return;
  const int s = threadIdx.x & (QR_MAX - 1), j4 = (st->base + 3) & ~3;
  const bool ok = s < st->r;
  const double* src = LT + (ok ? st->slot[s] : 0);
  constexpr int ROWS = 256 / QR_MAX;
  for (int q = blockIdx.x * ROWS + threadIdx.x / QR_MAX; q < j4; q += gridDim.x * ROWS)
    LP[q * QR_MAX + s] = ok ? src[(long)q * QC] : 0.0;
}

// The round's r columns of L for all points, one pass over the earlier ones:
// acc[s][a] = sum_q L[q][p_s] L[q][a] by MFMA (A: the pivots' entries from LP,
// B: 32 points a wave, two interleaved 16-point fragments from one 16-byte
// load), G the same way from the orbitals, then the triangular solve with one
// lane a point.  Even and odd steps of four are summed apart: with one chain
// |R_jj| was 2.5e-14 from the exact values on 40^3, K = 512, with two 2.1e-14 (one
// kernel per pivot: 2.0e-14).  Loads of QU steps are in flight while the previous
// QU are multiplied.  Bound by the read of L, 8 j N bytes a round, and by
// latency: two waves a SIMD at N = 64000, 3.4 TB/s.
constexpr int QU = 8;
constexpr int QW = QB / 32;  // waves of a workgroup: 32 points each, QB together

template <int G>
__global__ __launch_bounds__(64 * QW) void qr_apply(const double* __restrict__ phi, const double* __restrict__ occ,
                                                    long n, int m, int mo, double* __restrict__ d,
                                                    double* __restrict__ L, long ln, const double* __restrict__ LP,
                                                    const QrState* __restrict__ st, double* pv, int* pi, int* hist) {
  if (st->done || st->stall) return;
  __shared__ double tile[QW][32][QR_MAX + 1];
  __shared__ int h[QBINS];
  __shared__ double sv[QW];
  __shared__ int si[QW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l16 = lane & 15, l4 = lane >> 4;
  const int r = st->r, j = st->base;
  const bool two = r > 16;
  const long a0 = (long)blockIdx.x * QB + 32 * w;
  qd4 acc[2][2] = {}, odd[2][2] = {}, p1[2][2] = {}, p2[2][2] = {};
  {
    // rows are ln >= the workgroups' points apart, so every load is inside L
    const double2* lb = reinterpret_cast<const double2*>(L + (long)l4 * ln + a0 + 2 * l16);
    const double* t0 = LP + l4 * QR_MAX + l16;
    const long lstep = 2 * ln;  // four rows, in double2
    const int n4 = j >> 2;      // whole steps of four columns
    auto columns = [&](auto both) {
      double2 b[2][QU];
      double u0[2][QU], u1[2][QU];
      auto load = [&](int buf, int q0) {
#pragma unroll
        for (int u = 0; u < QU; ++u) {
          const int q = min(q0 + u, n4 - 1);
          b[buf][u] = lb[q * lstep];
          u0[buf][u] = t0[q * 4 * QR_MAX];
          if (both.value) u1[buf][u] = t0[q * 4 * QR_MAX + 16];
        }
      };
      auto mul = [&](int buf, int u) {
        auto& s = u & 1 ? odd : acc;
        s[0][0] = qr_mfma(u0[buf][u], b[buf][u].x, s[0][0]);
        s[0][1] = qr_mfma(u0[buf][u], b[buf][u].y, s[0][1]);
        if (both.value) {
          s[1][0] = qr_mfma(u1[buf][u], b[buf][u].x, s[1][0]);
          s[1][1] = qr_mfma(u1[buf][u], b[buf][u].y, s[1][1]);
        }
      };
      load(0, 0);
      int q = 0;
      for (; q + 2 * QU <= n4; q += 2 * QU) {
        load(1, q + QU);
#pragma unroll
        for (int u = 0; u < QU; ++u) mul(0, u);
        load(0, q + 2 * QU);  // past the end: the last step again, not multiplied
#pragma unroll
        for (int u = 0; u < QU; ++u) mul(1, u);
      }
      if (q + QU < n4) load(1, q + QU);
#pragma unroll
      for (int u = 0; u < 2 * QU; ++u)
        if (q + u < n4) mul(u / QU, u % QU);
    };
    if (n4 > 0) {
      if (two) columns(std::true_type{});
      else columns(std::false_type{});
    }
    if (j & 3) {  // the last one to three columns; LP is zero beyond them, L is not
      const bool ok = 4 * n4 + l4 < j;
      const double2 x = ok ? lb[n4 * lstep] : double2{0.0, 0.0};
      const double v0 = t0[n4 * 4 * QR_MAX], v1 = t0[n4 * 4 * QR_MAX + 16];
      acc[0][0] = qr_mfma(v0, x.x, acc[0][0]);
      acc[0][1] = qr_mfma(v0, x.y, acc[0][1]);
      acc[1][0] = qr_mfma(v1, x.x, acc[1][0]);
      acc[1][1] = qr_mfma(v1, x.y, acc[1][1]);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      acc[i][f] += odd[i][f];
      odd[i][f] = qd4{};
    }
  {
    const long ra = min(a0 + 2 * l16, n - 1), rb = min(a0 + 2 * l16 + 1, n - 1);
    const long q0 = st->piv[min(l16, r - 1)], q1 = st->piv[min(16 + l16, r - 1)];
    qd4 odd2[2][2] = {};
    auto four = [&](const double* __restrict__ rows, int width, int k, qd4(&s)[2][2], qd4(&si)[2][2]) {
      const bool ok = k < width;
      const double x = ok ? rows[ra * width + k] : 0.0, y = ok ? rows[rb * width + k] : 0.0;
      const double u = ok ? rows[q0 * width + k] : 0.0, v = ok ? rows[q1 * width + k] : 0.0;
      s[0][0] = qr_mfma(u, x, s[0][0]);
      s[0][1] = qr_mfma(u, y, s[0][1]);
      if (two) {
        s[1][0] = qr_mfma(v, x, s[1][0]);
        s[1][1] = qr_mfma(v, y, s[1][1]);
      }
      if (G == G_MODULUS) {
        const double u2 = ok ? qr_times_i(rows, q0, width, k) : 0.0;
        const double v2 = ok ? qr_times_i(rows, q1, width, k) : 0.0;
        si[0][0] = qr_mfma(u2, x, si[0][0]);
        si[0][1] = qr_mfma(u2, y, si[0][1]);
        si[1][0] = qr_mfma(v2, x, si[1][0]);
        si[1][1] = qr_mfma(v2, y, si[1][1]);
      }
    };
    for (int k0 = l4; k0 < m + l4; k0 += 8) {
      four(phi, m, k0, p1, p2);
      four(phi, m, k0 + 4, odd, odd2);
    }
    if (G == G_PRODUCT)
      for (int k0 = l4; k0 < mo + l4; k0 += 8) {
        four(occ, mo, k0, p2, p2);
        four(occ, mo, k0 + 4, odd2, odd2);
      }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        p1[i][f] += odd[i][f];
        p2[i][f] += odd2[i][f];
      }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        tile[w][2 * l16 + f][16 * i + l4 + 4 * v] = qr_combine<G>(p1[i][f][v], p2[i][f][v]) - acc[i][f][v];
  __syncthreads();
  const long a = a0 + lane;
  double v = -DBL_MAX;
  int vi = INT_MAX;
  if (lane < 32 && a < n) {
    double x[QR_MAX];
#pragma unroll
    for (int s = 0; s < QR_MAX; ++s) x[s] = tile[w][lane][s];
    double da = d[a];
#pragma unroll
    for (int s = 0; s < QR_MAX; ++s)
      if (s < r) {
        const double l = x[s] * st->rs[s];
        L[(j + s) * ln + a] = l;
#pragma unroll
        for (int q = s + 1; q < QR_MAX; ++q) x[q] -= l * st->tri[s][q];
        if (a == st->piv[s] || da == RETIRED) da = RETIRED;
        else da -= l * l;
      }
    d[a] = da;
    v = da;
    vi = (int)a;
  }
  qr_count(v, st->refkey, h, hist);
  for (int o = 32; o > 0; o >>= 1) {
    const double ov = __shfl_xor(v, o);
    const int oi = __shfl_xor(vi, o);
    if (wins(ov, oi, v, vi)) { v = ov; vi = oi; }
  }
  if (lane == 0) { sv[w] = v; si[w] = vi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < QW; ++q)
      if (wins(sv[q], si[q], v, vi)) { v = sv[q]; vi = si[q]; }
    pv[blockIdx.x] = v;
    pi[blockIdx.x] = vi;
  }
}

// ---- one pivot a step: complex half-rotated orbitals, few pivots, more equal points than candidates
// Pivot step j; partial maxima are read from (pv_in, pi_in) and written to
// (pv_out, pi_out), which the host alternates between steps.  G_COMPLEX: L is
// complex too, row 2q (ln doubles apart) holds the real, row 2q + 1 the
// imaginary parts of column q.
template <int G>
__global__ __launch_bounds__(QB) void qr_step(const double* __restrict__ phi, const double* __restrict__ occ, long n,
                                              int m, int mo, int j, int nparts, double* __restrict__ d,
                                              double* __restrict__ L, long ln, const double* pv_in, const int* pi_in,
                                              double* pv_out, int* pi_out, int* piv, double* rdiag, int* fail) {
  extern __shared__ double sh[];  // pivot rows: phi (m), occ (mo), then L[q][p], 2j values
  __shared__ double gv;
  __shared__ int gi;
  // global argmax of the previous residuals (every block, redundantly)
  {
    double v = -DBL_MAX;
    int vi = INT_MAX;
    for (int q = threadIdx.x; q < nparts; q += QB)
      if (wins(pv_in[q], pi_in[q], v, vi)) { v = pv_in[q]; vi = pi_in[q]; }
    for (int o = 32; o > 0; o >>= 1) {
      const double ov = __shfl_xor(v, o);
      const int oi = __shfl_xor(vi, o);
      if (wins(ov, oi, v, vi)) { v = ov; vi = oi; }
    }
    __shared__ double wv[QB / 64];
    __shared__ int wi[QB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) { wv[w] = v; wi[w] = vi; }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int q = 1; q < QB / 64; ++q)
        if (wins(wv[q], wi[q], v, vi)) { v = wv[q]; vi = wi[q]; }
      gv = v;
      gi = vi;
    }
    __syncthreads();
  }
  const double pval = gv;
  const long p = gi;
  // residual exhausted (K beyond the numerical rank): below 1e-13 of the first
  // pivot the squared residuals are rounding noise of the Gram downdate
  const double d0 = j > 0 ? rdiag[0] * rdiag[0] : pval;
  if (!(pval > 1e-13 * d0) || p < 0 || p >= n) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *fail = j + 1;
    return;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    piv[j] = (int)p;
    rdiag[j] = sqrt(pval);
  }
  double* prow = sh;
  double* orow = sh + m;
  double* lp = orow + (occ ? mo : 0);
  constexpr int LW = G == G_COMPLEX ? 2 : 1;  // doubles per entry of L
  for (int q = threadIdx.x; q < m; q += QB) prow[q] = phi[p * m + q];
  if (occ)
    for (int q = threadIdx.x; q < mo; q += QB) orow[q] = occ[p * mo + q];
  for (int q = threadIdx.x; q < LW * j; q += QB) lp[q] = L[q * ln + p];
  __syncthreads();
  const double rs = 1.0 / sqrt(pval);
  const long a = (long)blockIdx.x * QB + threadIdx.x;
  double v = -DBL_MAX;
  int vi = INT_MAX;
  if (a < n) {
    double da = d[a], lr, li = 0.0;
    if constexpr (G == G_COMPLEX) {
      double qr, qi, o_r, o_i;
      cdot_row(phi + a * m, prow, m, qr, qi);
      cdot_row(occ + a * mo, orow, mo, o_r, o_i);
      const double gr = o_r * qr + o_i * qi, gi = o_r * qi - o_i * qr;  // conj(Qocc) Q
      double ar = 0.0, ai = 0.0;
      for (int q = 0; q < j; ++q) {
        const double xr = L[2 * q * ln + a], xi = L[(2 * q + 1) * ln + a];
        const double yr = lp[2 * q], yi = lp[2 * q + 1];
        ar = fma(xr, yr, fma(xi, yi, ar));
        ai = fma(xi, yr, fma(-xr, yi, ai));
      }
      lr = (gr - ar) * rs;
      li = (gi - ai) * rs;
      L[2 * j * ln + a] = lr;
      L[(2 * j + 1) * ln + a] = li;
    } else {
      double g, h = 0.0;
      if constexpr (G == G_MODULUS) cdot_row(phi + a * m, prow, m, g, h);
      else g = dot_row(phi + a * m, prow, m);
      if constexpr (G == G_PRODUCT) h = dot_row(occ + a * mo, orow, mo);
      double s0 = 0.0, s1 = 0.0;
      int q = 0;
      for (; q + 2 <= j; q += 2) {
        s0 = fma(L[q * ln + a], lp[q], s0);
        s1 = fma(L[(q + 1) * ln + a], lp[q + 1], s1);
      }
      if (q < j) s0 = fma(L[q * ln + a], lp[q], s0);
      lr = (qr_combine<G>(g, h) - (s0 + s1)) * rs;
      L[j * ln + a] = lr;
    }
    if (a == p || da == RETIRED) da = RETIRED;
    else da -= lr * lr + li * li;
    d[a] = da;
    v = da;
    vi = (int)a;
  }
  block_argmax(v, vi, pv_out, pi_out);
}

}  // namespace

// L of the rounds: rows of whole workgroups' points
inline long qr_ln(long n) { return (n + QB - 1) / QB * QB; }

size_t qrcp_work_bytes(long n, int k, bool cplx) {
  const long nparts = (n + QB - 1) / QB;
  return carve_bytes<double>((size_t)n) + carve_bytes<double>((size_t)qr_ln(n) * k * (cplx ? 2 : 1)) +
         2 * carve_bytes<double>(nparts) + 2 * carve_bytes<int>(nparts) +
         carve_bytes<char>(sizeof(double) * k + sizeof(int) * ((size_t)k + 1)) + carve_bytes<double>((size_t)(k + 4) * QC) +
         carve_bytes<double>((size_t)(k + 4) * QR_MAX) + carve_bytes<double>((size_t)QC * QC) + carve_bytes<int>(QC) +
         carve_bytes<int>(QBINS) + carve_bytes<QrState>(1);
}

namespace {

// The orbitals, d, L and the maxima of a run; pv, pi [cur] are the latest.
struct QrRun {
  const double *phi, *occ;
  long n;
  int m, mo, k;
  double *d, *L, *pv[2];
  int* pi[2];
  double* rd;  // rd, piv and fail lie together: one copy back
  int *piv, *fail;
  int nparts;
  long ln;
  size_t lds;  // of a step, at most
};

// Pivot steps j .. j + count - 1; an even count leaves the latest maxima in [0].
template <int G>
int qr_steps(const QrRun& q, int j, int count, hipStream_t s) {
  if (q.lds > 64 * 1024)
    THC_HIP(hipFuncSetAttribute((const void*)qr_step<G>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)q.lds));
  for (int i = 0; i < count; ++i) {
    const int in = i & 1;
    hipLaunchKernelGGL(qr_step<G>, dim3((unsigned)q.nparts), dim3(QB), q.lds, s, q.phi, q.occ, q.n, q.m, q.mo, j + i,
                       q.nparts, q.d, q.L, q.ln, q.pv[in], q.pi[in], q.pv[in ^ 1], q.pi[in ^ 1], q.piv, q.rd, q.fail);
  }
  THC_HIP(hipGetLastError());
  return THC_OK;
}

// Rounds of pivots (real G) until k are chosen.
template <int G>
int qr_rounds(const QrRun& q, Arena& ws, hipStream_t s) {
  const int k = q.k;
  double* LT = ws.take<double>((size_t)(k + 4) * QC);
  double* LP = ws.take<double>((size_t)(k + 4) * QR_MAX);
  double* S = ws.take<double>((size_t)QC * QC);
  int* cand = ws.take<int>(QC);
  int* hist = ws.take<int>(QBINS);
  QrState* st = ws.take<QrState>(1);
  if (!LT || !LP || !S || !cand || !hist || !st) return THC_ERR_NO_MEMORY;
  auto begin = [&](int j) {
    hipLaunchKernelGGL(qr_begin, dim3(1), dim3(QB), 0, s, q.pv[0], q.pi[0], q.nparts, j, k, q.fail, st, hist);
    hipLaunchKernelGGL(qr_hist, dim3(q.nparts), dim3(QB), 0, s, q.d, q.n, st, hist);
  };
  begin(0);
  // Every round chooses a pivot, ends the run or stalls.  The host looks after
  // up to eight rounds, fewer where the pivots left should take fewer (16 a
  // round) or a round stalled lately; rounds past an end or a stall return at
  // once.
  int h[3] = {0, 0, 0};  // j, done, stall
  int steps = 4, most = 8;
  while (!h[1]) {
    const int batch = std::min(most, (k - h[0] + 15) / 16);
    for (int b = 0; b < batch; ++b) {
      hipLaunchKernelGGL(qr_pick, dim3(q.nparts), dim3(QB), 0, s, q.d, q.n, hist, st, cand);
      hipLaunchKernelGGL(qr_gather, dim3(256), dim3(QC), 0, s, q.L, q.ln, st, cand, LT);
      hipLaunchKernelGGL(qr_gram<G>, dim3((QC / 16) * (QC / 16)), dim3(256), 0, s, q.phi, q.occ, q.m, q.mo, st, cand, LT,
                         S);
      hipLaunchKernelGGL(qr_run, dim3(1), dim3(1024), 0, s, S, q.d, cand, k, st, hist, q.piv, q.rd, q.fail);
      hipLaunchKernelGGL(qr_compact, dim3(64), dim3(256), 0, s, st, LT, LP);
      hipLaunchKernelGGL(qr_apply<G>, dim3(q.nparts), dim3(64 * QW), 0, s, q.phi, q.occ, q.n, q.m, q.mo, q.d, q.L, q.ln,
                         LP, st, q.pv[0], q.pi[0], hist);
    }
    THC_HIP(hipGetLastError());
    const int before = h[0];
    THC_HIP(hipMemcpyAsync(h, &st->j, sizeof(h), hipMemcpyDeviceToHost, s));
    THC_HIP(hipStreamSynchronize(s));
    most = std::min(8, 2 * most);
    if (h[0] > before) steps = std::max(4, steps / 2);
    if (h[1] || !h[2]) continue;
    const int count = std::min(steps, k - h[0]);
    THC_TRY(qr_steps<G>(q, h[0], count, s));
    h[0] += count;
    begin(h[0]);
    steps = std::min(32, 2 * steps);
    most = 1;
  }
  return THC_OK;
}

template <int G>
int qr_run_all(const QrRun& q, bool by_steps, Arena& ws, hipStream_t s) {
  if constexpr (G != G_COMPLEX)
    if (!by_steps) return qr_rounds<G>(q, ws, s);
  THC_HIP(hipMemsetAsync(q.fail, 0, sizeof(int), s));
  return qr_steps<G>(q, 0, q.k, s);
}

}  // namespace

int qrcp_points(const double* phi, const double* occ, long n, int m, int mo, int k, int* piv_out, double* rdiag_out,
                Arena& ws, hipStream_t s, bool cplx) {
  const long nparts = (n + QB - 1) / QB;
  if (nparts > 0x7fffffffL) return THC_ERR_ARG;
  if (cplx && (m % 2 || (occ && mo % 2))) return THC_ERR_ARG;
  const int g = cplx ? (occ ? G_COMPLEX : G_MODULUS) : (occ ? G_PRODUCT : G_SQUARE);
  const int lw = g == G_COMPLEX ? 2 : 1;
  QrRun q = {phi, occ, n, m, occ ? mo : 0, k};
  q.nparts = (int)nparts;
  q.ln = qr_ln(n);
  q.d = ws.take<double>((size_t)n);
  q.L = ws.take<double>((size_t)q.ln * k * lw);
  for (int i = 0; i < 2; ++i) {
    q.pv[i] = ws.take<double>(nparts);
    q.pi[i] = ws.take<int>(nparts);
  }
  const size_t back = sizeof(double) * k + sizeof(int) * ((size_t)k + 1);
  char* result = ws.take<char>(back);
  q.rd = reinterpret_cast<double*>(result);
  q.piv = reinterpret_cast<int*>(q.rd + k);
  q.fail = q.piv + k;
  if (!q.d || !q.L || !q.pv[0] || !q.pv[1] || !q.pi[0] || !q.pi[1] || !result) return THC_ERR_NO_MEMORY;
  q.lds = sizeof(double) * ((size_t)m + q.mo + (size_t)k * lw);
  if (q.lds > 160 * 1024) return THC_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(qr_init, dim3((unsigned)nparts), dim3(QB), 0, s, phi, occ, n, m, mo, q.d, q.pv[0], q.pi[0]);
  THC_HIP(hipGetLastError());
  // Few pivots: a step is 8 us on a small grid and a round of shared pivots 75,
  // of which six or seven are taken whatever k (27^3 points, k = 54: 0.44 ms in
  // steps, 0.47 in rounds; 32^3 points, k = 50: 0.44 and 0.53; but 32^3 points,
  // k = 67: 0.58 and 0.41; 48^3 points, k = 40: 0.67 and 0.33).  Steps of complex
  // orbitals cost more (24^3 points, M = 16: k = 8 0.14 both, k = 16 0.20 and
  // 0.16).  Up to four pivots take less than what surrounds one round (48^3
  // points, k = 2: 0.09 and 0.15; k = 4: 0.12 and 0.16; 64^3 points, M = 100,
  // k = 1: 0.23 and 0.28, k = 2: 0.28 both).
  const bool by_steps =
      k == 1 || (k <= 4 && n <= 120000) || (n <= 40000 && k < (g == G_MODULUS ? 9 : 64));
  switch (g) {
    case G_COMPLEX: THC_TRY(qr_run_all<G_COMPLEX>(q, true, ws, s)); break;
    case G_MODULUS: THC_TRY(qr_run_all<G_MODULUS>(q, by_steps, ws, s)); break;
    case G_PRODUCT: THC_TRY(qr_run_all<G_PRODUCT>(q, by_steps, ws, s)); break;
    default: THC_TRY(qr_run_all<G_SQUARE>(q, by_steps, ws, s));
  }
  std::vector<double> host((back + sizeof(double) - 1) / sizeof(double));
  THC_HIP(hipMemcpyAsync(host.data(), result, back, hipMemcpyDeviceToHost, s));
  THC_HIP(hipStreamSynchronize(s));
  const int* hp = reinterpret_cast<const int*>(host.data() + k);
  if (rdiag_out) std::copy(host.begin(), host.begin() + k, rdiag_out);
  if (hp[k]) return THC_ERR_NOT_POSDEF;
  std::vector<int> h(hp, hp + k);
  // the reference keeps the first K pivots in ascending grid order
  std::sort(h.begin(), h.end());
  THC_HIP(hipMemcpyAsync(piv_out, h.data(), sizeof(int) * k, hipMemcpyHostToDevice, s));
  THC_HIP(hipStreamSynchronize(s));
  return THC_OK;
}

}  // namespace thc
