// Weighted k-means (centroidal Voronoi) interpolation points on gfx950,
// bit-identical to the reference's sequential FP64 loop (src/kmeans.cpp).
//
// Exactness rules kept by every kernel here:
//  * distances are sqrt((dx*dx + dy*dy) + dz*dz) with dx = centroid - point,
//    every multiply and add rounded separately (no FMA contraction, below), and
//    sqrt correctly rounded (the device sqrt is; tests check it);
//  * the argmin takes the first index among equal rounded distances
//    (std::min_element), evaluated as a lexicographic (distance, index) minimum;
//    sqrt is monotone, so a sqrt is only needed when d^2 improves;
//  * centroid sums run per cluster in ascending grid index with the product
//    rounded before the add (a bitmap over the members' indices supplies that
//    order), and are divided once (IEEE double division);
//  * pruning of centroids (or grid tiles) is conservative: a candidate is
//    dropped only if its distance bound exceeds the best bound by a relative
//    1e-8 on squares, far above the few-ulp rounding of any distance.
#pragma clang fp contract(off)
#include <atomic>
#include <cfloat>
#include <climits>
#include <type_traits>
#include <vector>

#include "common.h"
#include "kmeans.h"

namespace thc {
namespace km {

__device__ inline double dist2(double cx, double cy, double cz, double gx, double gy, double gz) {
  const double dx = cx - gx;
  const double dy = cy - gy;
  const double dz = cz - gz;
  return (dx * dx + dy * dy) + dz * dz;
}

// Lexicographic (rounded distance, index) update for candidates visited in
// any order.  bd2 is the exact d^2 of the current best.
__device__ inline void consider_any(double d2, int idx, double& bd2, double& bs, int& bi) {
  if (d2 < bd2) {
    const double s = sqrt(d2);
    if (s < bs || (s == bs && idx < bi)) { bs = s; bd2 = d2; bi = idx; }
  } else if (d2 == bd2) {
    if (idx < bi) bi = idx;
  } else if (idx < bi && d2 <= bd2 * (1.0 + 0x1p-50)) {
    // d^2 slightly above the best may still round to the same distance
    const double s = sqrt(d2);
    if (s == bs) bi = idx;
  }
}

__device__ inline double lb2_box(double cx, double cy, double cz, const double* b) {
  const double gx = fmax(0.0, fmax(b[0] - cx, cx - b[3]));
  const double gy = fmax(0.0, fmax(b[1] - cy, cy - b[4]));
  const double gz = fmax(0.0, fmax(b[2] - cz, cz - b[5]));
  return gx * gx + gy * gy + gz * gz;
}
__device__ inline double ub2_box(double cx, double cy, double cz, const double* b) {
  const double ex = fmax(fabs(cx - b[0]), fabs(cx - b[3]));
  const double ey = fmax(fabs(cy - b[1]), fabs(cy - b[4]));
  const double ez = fmax(fabs(cz - b[2]), fabs(cz - b[5]));
  return ex * ex + ey * ey + ez * ez;
}
constexpr double PRUNE = 1.0 + 1e-8;

// Wave-wide reductions by DPP moves: within rows of 16 lanes by shifts, then
// lane 15 of a row into the next row and lane 31 into the upper half, so lane
// 63 ends with the result (about 25 cycles a step; a cross-lane permute through
// LDS takes over 100).  Every lane of the wave must be active.
template <int CTRL, int ROWS>
__device__ inline double dpp_min(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return fmin(v, __longlong_as_double(((long long)hi << 32) | (unsigned)lo));
}
__device__ inline double wave_min(double v) {
  v = dpp_min<0x111, 0xf>(v);
  v = dpp_min<0x112, 0xf>(v);
  v = dpp_min<0x114, 0xf>(v);
  v = dpp_min<0x118, 0xf>(v);
  v = dpp_min<0x142, 0xa>(v);
  v = dpp_min<0x143, 0xc>(v);
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int CTRL, int ROWS>
__device__ inline int dpp_get(int none, int v) { return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false); }
// inclusive sum over the lanes up to this one
__device__ inline int wave_scan(int v) {
  v += dpp_get<0x111, 0xf>(0, v);
  v += dpp_get<0x112, 0xf>(0, v);
  v += dpp_get<0x114, 0xf>(0, v);
  v += dpp_get<0x118, 0xf>(0, v);
  v += dpp_get<0x142, 0xa>(0, v);
  v += dpp_get<0x143, 0xc>(0, v);
  return v;
}
__device__ inline int wave_sum(int v) { return __builtin_amdgcn_readlane(wave_scan(v), 63); }
__device__ inline int wave_min(int v) {
  v = min(v, dpp_get<0x111, 0xf>(v, v));
  v = min(v, dpp_get<0x112, 0xf>(v, v));
  v = min(v, dpp_get<0x114, 0xf>(v, v));
  v = min(v, dpp_get<0x118, 0xf>(v, v));
  v = min(v, dpp_get<0x142, 0xa>(v, v));
  v = min(v, dpp_get<0x143, 0xc>(v, v));
  return __builtin_amdgcn_readlane(v, 63);
}

// acc + v[0] + v[1] + ... strictly left to right (one lane's chain), from LDS
// at 16-byte alignment: the next sixteen terms are read while the current ones
// are added.
__device__ inline double seq_sum(double acc, const double* v, int len) {
  const double2* p = reinterpret_cast<const double2*>(v);
  const int nb = len / 16;
  double2 a[8], b[8];
  if (nb > 0) {
#pragma unroll
    for (int q = 0; q < 8; ++q) a[q] = p[q];
  }
  for (int i = 0; i < nb; i += 2) {
    const int i1 = min(i + 1, nb - 1), i2 = min(i + 2, nb - 1);
#pragma unroll
    for (int q = 0; q < 8; ++q) b[q] = p[8 * i1 + q];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      acc += a[q].x;
      acc += a[q].y;
    }
    if (i + 1 >= nb) break;
#pragma unroll
    for (int q = 0; q < 8; ++q) a[q] = p[8 * i2 + q];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      acc += b[q].x;
      acc += b[q].y;
    }
  }
  for (int i = 16 * nb; i < len; ++i) acc += v[i];
  return acc;
}

// ------------------------------------------------------------------ setup

__device__ __forceinline__ void bbox_partial_b(const double* grid, long n, double* part, int bid, int nblk) {
  double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  for (long i = bid * 256L + threadIdx.x; i < n; i += 256L * nblk)
    for (int d = 0; d < 3; ++d) {
      const double v = grid[i * 3 + d];
      lo[d] = fmin(lo[d], v);
      hi[d] = fmax(hi[d], v);
    }
  __shared__ double s[6][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int d = 0; d < 3; ++d) {
    double a = wave_min(lo[d]), b = -wave_min(-hi[d]);
    if (lane == 0) { s[d][w] = a; s[3 + d][w] = b; }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int d = threadIdx.x;
    double r = s[d][0];
    for (int q = 1; q < 4; ++q) r = d < 3 ? fmin(r, s[d][q]) : fmax(r, s[d][q]);
    part[bid * 6 + d] = r;
  }
}
__global__ __launch_bounds__(256) void bbox_partial(const double* grid, long n, double* part) {
  bbox_partial_b(grid, n, part, (int)blockIdx.x, (int)gridDim.x);
}

__device__ inline unsigned spread3(unsigned v) {
  unsigned r = 0;
  for (int b = 0; b < 10; ++b) r |= ((v >> b) & 1u) << (3 * b);
  return r;
}

// Morton cell of every point inside the bounding box of the nb partial ones
// (nb <= 256; every workgroup folds them by itself).
__device__ __forceinline__ void morton_keys_b(const double* grid, long n, const double* part, int nb, int cells,
                                                   int* keys, int bid) {
  __shared__ double s[6][4];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  for (int d = 0; d < 3; ++d) {
    const double a = wave_min(t < nb ? part[t * 6 + d] : DBL_MAX);
    const double b = -wave_min(t < nb ? -part[t * 6 + 3 + d] : DBL_MAX);
    if (lane == 0) { s[d][w] = a; s[3 + d][w] = b; }
  }
  __syncthreads();
  const long i = bid * 256L + t;
  if (i >= n) return;
  unsigned c[3];
  for (int d = 0; d < 3; ++d) {
    const double lo = fmin(fmin(s[d][0], s[d][1]), fmin(s[d][2], s[d][3]));
    const double ext = fmax(fmax(s[3 + d][0], s[3 + d][1]), fmax(s[3 + d][2], s[3 + d][3])) - lo;
    int v = 0;
    if (ext > 0) v = (int)((grid[i * 3 + d] - lo) / ext * cells);
    c[d] = (unsigned)min(max(v, 0), cells - 1);
  }
  keys[i] = (int)((spread3(c[0]) << 2) | (spread3(c[1]) << 1) | spread3(c[2]));
}
__global__ __launch_bounds__(256) void morton_keys(const double* grid, long n, const double* part, int nb, int cells,
                                                   int* keys) {
  morton_keys_b(grid, n, part, nb, cells, keys, (int)blockIdx.x);
}

// The sorted coordinates, the bounding box of each tile of TP of them and
// those of its four runs of 64 (one wave of the assignment each).
__device__ __forceinline__ void sorted_tiles_b(const double* grid, const int* perm, long n, double* sx, double* sy,
                                                    double* sz, double* boxes, double* wboxes, int bid) {
  const long p = bid * (long)TP + threadIdx.x;
  double v[3] = {0, 0, 0};
  const bool ok = p < n;
  if (ok) {
    const long i = perm[p];
    for (int d = 0; d < 3; ++d) v[d] = grid[i * 3 + d];
    sx[p] = v[0];
    sy[p] = v[1];
    sz[p] = v[2];
  }
  __shared__ double s[6][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int d = 0; d < 3; ++d) {
    const double a = wave_min(ok ? v[d] : DBL_MAX), b = -wave_min(ok ? -v[d] : DBL_MAX);
    if (lane == 0) { s[d][w] = a; s[3 + d][w] = b; }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int d = threadIdx.x;
    double r = s[d][0];
    for (int q = 1; q < 4; ++q) r = d < 3 ? fmin(r, s[d][q]) : fmax(r, s[d][q]);
    boxes[bid * 6 + d] = r;
  }
  if (threadIdx.x < 24) wboxes[bid * 24L + threadIdx.x] = s[threadIdx.x % 6][threadIdx.x / 6];
}
__global__ __launch_bounds__(256) void sorted_tiles(const double* grid, const int* perm, long n, double* sx, double* sy,
                                                    double* sz, double* boxes, double* wboxes) {
  sorted_tiles_b(grid, perm, n, sx, sy, sz, boxes, wboxes, (int)blockIdx.x);
}

// Start of a run: the loop state, the starting centroids, empty buckets and
// lists (ctr) and change counts.
__device__ __forceinline__ void init_run_b(const double* grid, const int* idx, int k, double* cen, int* cnt, int* ctr,
                                                int* chg, int nchg, State* st, int bid, int nblk) {
  const int j = bid * 256 + threadIdx.x;
  if (ctr && j < 4) ctr[j] = 0;
  for (int i = j; i < nchg; i += nblk * 256) chg[i] = 0;
  if (j == 0) {
    st->ended = INT_MAX;
    st->final_buf = 0;
    st->error = 0;
    st->bad = INT_MAX;
    st->iters = 0;
    st->mode = MODE_LATEST;
    st->dups = 0;
    st->last_diff = 0.0;
  }
  if (j >= k) return;
  if (cnt) cnt[j] = 0;
  if (!idx) return;
  const long i = idx[j];
  cen[j * 3 + 0] = grid[i * 3 + 0];
  cen[j * 3 + 1] = grid[i * 3 + 1];
  cen[j * 3 + 2] = grid[i * 3 + 2];
}
__global__ __launch_bounds__(256) void init_run(const double* grid, const int* idx, int k, double* cen, int* cnt,
                                                int* ctr, int* chg, int nchg, State* st) {
  init_run_b(grid, idx, k, cen, cnt, ctr, chg, nchg, st, (int)blockIdx.x, (int)gridDim.x);
}

// ------------------------------------------------------------------ stable counting sort (Morton cells)

// Per index-order tile of CS_TILE points: histogram of keys.
__device__ __forceinline__ void cs_hist_b(const int* keys, long n, int nbins, int* tile_count, int bid, int nblk) {
  __shared__ int h[MAXB];
  for (int b = threadIdx.x; b < nbins; b += 256) h[b] = 0;
  __syncthreads();
  const long base = (long)bid * CS_TILE;
  for (int e = threadIdx.x; e < CS_TILE; e += 256) {
    const long i = base + e;
    if (i < n) {
      const int key = keys[i];
      if ((unsigned)key < (unsigned)nbins) atomicAdd(&h[key], 1);
    }
  }
  __syncthreads();
  int* out = tile_count + (long)bid * nbins;
  for (int b = threadIdx.x; b < nbins; b += 256) out[b] = h[b];
}
__global__ __launch_bounds__(256) void cs_hist(const int* keys, long n, int nbins, int* tile_count) {
  cs_hist_b(keys, n, nbins, tile_count, (int)blockIdx.x, (int)gridDim.x);
}

// Column scan over tiles, in place: tile_count[t][b] -> exclusive offset of
// tile t within bin b; total[b] = count of bin b.  A workgroup takes 64 bins;
// its CS_SCAN_W waves scan consecutive runs of the tiles, then add the earlier
// runs' totals (16 waves: two dependent load rounds per wave at 256 tiles,
// where 4 waves needed eight).
__device__ __forceinline__ void cs_colscan_b(int* tile_count, int ntiles, int nbins, int* total, int bid, int nblk) {
  __shared__ int part[CS_SCAN_W][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b = bid * 64 + lane;
  const int per = (ntiles + CS_SCAN_W - 1) / CS_SCAN_W;
  const int t0 = wave * per, t1 = min(ntiles, t0 + per);
  // chunks of 16 tiles: every load of a chunk is issued before its first use
  // and before the chunk's stores (on this target stores and loads share one
  // completion counter, so a load after a store would wait for the store)
  constexpr int CH = 16;
  int run = 0;
  if (b < nbins)
    for (int t = t0; t < t1; t += CH) {
      int c[CH];
#pragma unroll
      for (int q = 0; q < CH; ++q) c[q] = (t + q < t1) ? tile_count[(long)(t + q) * nbins + b] : 0;
#pragma unroll
      for (int q = 0; q < CH; ++q) run += c[q];
    }
  part[wave][lane] = run;
  __syncthreads();
  int off = 0;
  for (int w = 0; w < wave; ++w) off += part[w][lane];
  if (b < nbins) {
    for (int t = t0; t < t1; t += CH) {
      int c[CH];
#pragma unroll
      for (int q = 0; q < CH; ++q) c[q] = (t + q < t1) ? tile_count[(long)(t + q) * nbins + b] : 0;
#pragma unroll
      for (int q = 0; q < CH; ++q)
        if (t + q < t1) {
          tile_count[(long)(t + q) * nbins + b] = off;
          off += c[q];
        }
    }
    if (wave == CS_SCAN_W - 1) total[b] = off;
  }
}
__global__ __launch_bounds__(64 * CS_SCAN_W) void cs_colscan(int* tile_count, int ntiles, int nbins, int* total) {
  cs_colscan_b(tile_count, ntiles, nbins, total, (int)blockIdx.x, (int)gridDim.x);
}

// Exclusive scan of total[0..nbins) into start (one workgroup of 1024).
__device__ __forceinline__ void cs_totscan_b(const int* total, int nbins, int* start, int bid, int nblk) {
  __shared__ int s[1024];
  const int t = threadIdx.x;
  const int per = (nbins + 1023) / 1024;
  int loc = 0;
  for (int q = 0; q < per; ++q) {
    const int b = t * per + q;
    if (b < nbins) loc += total[b];
  }
  s[t] = loc;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int v = t >= off ? s[t - off] : 0;
    __syncthreads();
    s[t] += v;
    __syncthreads();
  }
  int run = s[t] - loc;  // exclusive
  for (int q = 0; q < per; ++q) {
    const int b = t * per + q;
    if (b < nbins) {
      start[b] = run;
      run += total[b];
    }
  }
}
__global__ __launch_bounds__(1024) void cs_totscan(const int* total, int nbins, int* start) {
  cs_totscan_b(total, nbins, start, (int)blockIdx.x, (int)gridDim.x);
}

// Stable scatter: out[start[key] + rank] = index, rank counting earlier
// indices with the same key.  Chunks of 256 go in order; inside a chunk the
// four waves go in order; inside a wave, lanes with equal keys are ranked by
// lane through a 'nbits'-ballot match.
__device__ __forceinline__ void cs_scatter_b(const int* keys, long n, int nbins, int nbits,
                                                  const int* tile_off, const int* start, int* out, int bid, int nblk) {
  __shared__ int cnt[MAXB];
  __shared__ int slot[256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int* toff = tile_off + (long)bid * nbins;
  for (int b = tid; b < nbins; b += 256) cnt[b] = start[b] + toff[b];
  __syncthreads();
  const long base = (long)bid * CS_TILE;
  for (int ch = 0; ch < CS_TILE / 256; ++ch) {
    const long i = base + ch * 256 + tid;
    int key = i < n ? keys[i] : 0;
    const bool valid = i < n && (unsigned)key < (unsigned)nbins;
    if (!valid) key = 0;
    unsigned long long peers = __ballot(valid);
    for (int bit = 0; bit < nbits; ++bit) {
      const bool on = (key >> bit) & 1;
      const unsigned long long bal = __ballot(valid && on);
      peers &= on ? bal : ~bal;
    }
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int rank = __popcll(peers & below);
    const int leader = valid ? (__ffsll((long long)peers) - 1) : 0;
    for (int w = 0; w < 4; ++w) {
      if (wave == w && valid && rank == 0) {
        const int b0 = cnt[key];
        cnt[key] = b0 + __popcll(peers);
        slot[tid] = b0;
      }
      __syncthreads();
    }
    if (valid) out[slot[wave * 64 + leader] + rank] = (int)i;
    __syncthreads();
  }
}
__global__ __launch_bounds__(256) void cs_scatter(const int* keys, long n, int nbins, int nbits,
                                                  const int* tile_off, const int* start, int* out) {
  cs_scatter_b(keys, n, nbins, nbits, tile_off, start, out, (int)blockIdx.x, (int)gridDim.x);
}

// ------------------------------------------------------------------ Lloyd iteration

// Nearest centroid of the TP points of one tile.
//
// Centroids whose distance bound to the tile's box exceeds the best upper
// bound are dropped; the others (about 40 at 256 points a cluster) are listed
// in ascending index.  Every wave drops those that its own 64 points' box
// excludes (about a third is left), and its points scan the rest.  The winner is the first
// index of the smallest rounded distance, but the scan compares squares: one
// below the best by a relative 2^-50 has a strictly smaller rounded root (the
// roots differ by more than 2^-52, two roundings by less), one not below the
// best has no smaller root, and only a group of candidates with a square in
// between takes the roots themselves.  N = 262144, K = 1024: 14 us, 4 of them
// the buckets, most of it latency (four waves a SIMD, each a chain of some ten
// loads, reductions and barriers).  With a root whenever any lane improved and
// the whole list for every wave it took 38 us.
//
// With buckets (cnt, bucket) the points of a cluster are also listed for
// centroid_sums in any order, one device atomic per tile and cluster that has
// points there: cap of them in its bucket, any more in one list of (cluster,
// point) for all clusters, over.  ctr: its length and that of centroid_sums'
// partitions, each for even and odd iterations; an iteration clears those of
// the next, which the one before it has used up.
constexpr double SURE = 1.0 + 0x1p-49;

// Point 'orig' as member number 'at' of its cluster, by every lane of a wave.
__device__ __forceinline__ void list_member(bool live, int cluster, int at, int orig, int* bucket, int cap, int2* over,
                                            int* nover) {
  if (live && at < cap) bucket[(long)cluster * cap + at] = orig;
  const unsigned long long more = __ballot(live && at >= cap);
  if (more) {
    const int lane = threadIdx.x & 63, first = __ffsll((long long)more) - 1;
    int base = 0;
    if (lane == first) base = atomicAdd(nover, __popcll(more));
    base = __shfl(base, first);
    if (live && at >= cap) over[base + __popcll(more & ((1ull << lane) - 1))] = make_int2(cluster, orig);
  }
}

//
// CPT: centroids a thread looks at (k <= 256 CPT); the smallest that holds k
// keeps the unrolled loops, their registers and the list short (K = 1024:
// 18 us with 16 for every k).
template <int CPT>
__device__ __forceinline__ void assign_b(const double* sx, const double* sy, const double* sz,
                                              const int* perm, long n, const double* boxes, const double* wboxes,
                                              const double* cen, int k, int* map_new, const int* map_old,
                                              int* cnt, int* bucket, int cap, int2* over, int* ctr, int* chg,
                                              const State* st, int it, int seen, int bid) {
  if (st && (st->ended <= seen || st->bad < it)) return;
  __shared__ int cidx[256 * CPT];
  __shared__ double ccx[CAND_CAP], ccy[CAND_CAP], ccz[CAND_CAP];
  __shared__ int lcnt[CAND_CAP], lbase[CAND_CAP];
  __shared__ double redd[4];
  __shared__ int redi[64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const double* b = boxes + (long)bid * 6;
  double box[6], wbox[6];
  for (int d = 0; d < 6; ++d) {
    box[d] = b[d];
    wbox[d] = wboxes[((long)bid * 4 + wave) * 6 + d];
  }
  const long p = (long)bid * TP + tid;
  const bool live = p < n;
  double gx = 0.0, gy = 0.0, gz = 0.0;
  int orig = 0, old = -1;
  if (live) {
    gx = sx[p];
    gy = sy[p];
    gz = sz[p];
    orig = perm[p];
    if (map_old) old = map_old[p];
  }

  // this thread's centroids j = q * 256 + tid, loaded once
  static_assert(CPT * 4 <= 64, "one count per lane in the scan of the lists");
  double rx[CPT], ry[CPT], rz[CPT];
#pragma unroll
  for (int q = 0; q < CPT; ++q) {
    const int j = q * 256 + tid;
    const bool ok = j < k;
    rx[q] = ok ? cen[j * 3] : 0.0;
    ry[q] = ok ? cen[j * 3 + 1] : 0.0;
    rz[q] = ok ? cen[j * 3 + 2] : 0.0;
  }
  double u = DBL_MAX;
#pragma unroll
  for (int q = 0; q < CPT; ++q)
    if (q * 256 + tid < k) u = fmin(u, ub2_box(rx[q], ry[q], rz[q], box));
  u = wave_min(u);
  if (lane == 0) redd[wave] = u;
  for (int c = tid; c < CAND_CAP; c += TP) lcnt[c] = 0;
  __syncthreads();
  u = fmin(fmin(redd[0], redd[1]), fmin(redd[2], redd[3]));
  const double thr = u * PRUNE;

  // ascending list: counts per (q, wave), one scan of the 64 counts, one store
  unsigned flags = 0;
#pragma unroll
  for (int q = 0; q < CPT; ++q) {
    int have = 0;
    if (q * 256 < k) {  // uniform over the workgroup
      const bool flag = q * 256 + tid < k && lb2_box(rx[q], ry[q], rz[q], box) <= thr;
      flags |= flag ? 1u << q : 0u;
      have = __popcll(__ballot(flag));
    }
    if (lane == 0) redi[q * 4 + wave] = have;
  }
  __syncthreads();
  const int mine = lane < CPT * 4 ? redi[lane] : 0, upto = wave_scan(mine);
  const int ncand = __builtin_amdgcn_readlane(upto, 63);
#pragma unroll
  for (int q = 0; q < CPT; ++q) {
    if (q * 256 >= k) break;
    const bool flag = (flags >> q) & 1;
    const unsigned long long bal = __ballot(flag);
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int off = __builtin_amdgcn_readlane(upto - mine, q * 4 + wave) + __popcll(bal & below);
    if (flag) {
      cidx[off] = q * 256 + tid;
      if (off < CAND_CAP) { ccx[off] = rx[q]; ccy[off] = ry[q]; ccz[off] = rz[q]; }
    }
  }
  __syncthreads();

  // this wave's own bound over the listed candidates
  const int cached = min(ncand, CAND_CAP);
  double wu = DBL_MAX;
  for (int c = lane; c < cached; c += 64) wu = fmin(wu, ub2_box(ccx[c], ccy[c], ccz[c], wbox));
  const double wthr = wave_min(wu) * PRUNE;

  // best candidate so far, by position in the list
  int bc = 0;
  double bd2 = 0.0;
  bool first = true;
  auto rooted = [&](double d2, int c) {  // the rule on rounded distances itself
    if (d2 < bd2 && sqrt(d2) < sqrt(bd2)) {
      bd2 = d2;
      bc = c;
    }
  };
  // eight candidates' distances at a time (their LDS reads in flight together);
  // the last group repeats its last candidate, which changes nothing
  constexpr int U = 8;
  for (int c0 = 0; c0 < cached; c0 += 64) {
    const int cl = c0 + lane;
    unsigned long long left =
        __ballot(cl < cached && lb2_box(ccx[cl & (CAND_CAP - 1)], ccy[cl & (CAND_CAP - 1)], ccz[cl & (CAND_CAP - 1)], wbox) <= wthr);
    while (left) {
      int at[U];
#pragma unroll
      for (int q = 0; q < U; ++q) {
        at[q] = left ? c0 + __ffsll((long long)left) - 1 : at[q > 0 ? q - 1 : 0];
        left &= left - 1;
      }
      double d2v[U];
#pragma unroll
      for (int q = 0; q < U; ++q) d2v[q] = dist2(ccx[at[q]], ccy[at[q]], ccz[at[q]], gx, gy, gz);
      if (first) {
        bd2 = d2v[0];
        bc = at[0];
        first = false;
      }
      double nd2 = bd2;
      int nc = bc;
      bool close = false;
#pragma unroll
      for (int q = 0; q < U; ++q) {
        const bool sure = d2v[q] * SURE <= nd2 && d2v[q] < nd2;
        close |= d2v[q] < nd2 && !sure;
        nd2 = sure ? d2v[q] : nd2;
        nc = sure ? at[q] : nc;
      }
      if (close) {
#pragma unroll
        for (int q = 0; q < U; ++q) rooted(d2v[q], at[q]);
      } else {
        bd2 = nd2;
        bc = nc;
      }
    }
  }
  if (first) bd2 = dist2(ccx[0], ccy[0], ccz[0], gx, gy, gz);
  int c = cached;
  for (; c < ncand; ++c) {
    double cx, cy, cz;
    if (c < CAND_CAP) { cx = ccx[c]; cy = ccy[c]; cz = ccz[c]; }
    else { const int j = cidx[c]; cx = cen[j * 3]; cy = cen[j * 3 + 1]; cz = cen[j * 3 + 2]; }
    rooted(dist2(cx, cy, cz, gx, gy, gz), c);
  }
  const int bj = cidx[bc];
  if (!bucket) {  // one classification: the map in grid order
    if (live) map_new[orig] = bj;
    return;
  }
  int rank = 0;
  if (live) {
    map_new[p] = bj;
    if (bc < CAND_CAP) rank = atomicAdd(&lcnt[bc], 1);
  }
  const int changed = wave_sum(live && map_old && old != bj ? 1 : 0);
  if (lane == 0) redi[wave] = changed;
  __syncthreads();
  for (int q = tid; q < cached; q += TP) {
    const int m = lcnt[q];
    if (m) lbase[q] = atomicAdd(&cnt[cidx[q]], m);
  }
  if (tid == 0 && map_old) {
    const int sum = redi[0] + redi[1] + redi[2] + redi[3];
    if (sum) atomicAdd(&chg[bid % CHG], sum);
  }
  if (bid == 0 && tid < 2) ctr[2 * tid + ((it + 1) & 1)] = 0;
  __syncthreads();
  const int at = !live ? 0 : (bc < CAND_CAP ? lbase[bc] + rank : atomicAdd(&cnt[bj], 1));
  list_member(live, bj, at, orig, bucket, cap, over, &ctr[it & 1]);
}
template <int CPT>
__global__ __launch_bounds__(256) void assign(const double* sx, const double* sy, const double* sz,
                                              const int* perm, long n, const double* boxes, const double* wboxes,
                                              const double* cen, int k, int* map_new, const int* map_old, int* cnt,
                                              int* bucket, int cap, int2* over, int* ctr, int* chg, const State* st,
                                              int it, int seen) {
  assign_b<CPT>(sx, sy, sz, perm, n, boxes, wboxes, cen, k, map_new, map_old, cnt, bucket, cap, over, ctr, chg, st, it,
                seen, (int)blockIdx.x);
}

// Buckets of an assignment given in grid order, CS_TILE points a workgroup;
// st->error: a key outside [0, k).  The points of a cluster are counted in LDS
// and take their places with one device atomic per tile and cluster: with one
// per point, 4096 points to each of 64 addresses queued for 1.3 ms (64^3, K 64).
__global__ __launch_bounds__(256) void bucket_map(const int* map, long n, int k, int* cnt, int* bucket, int cap,
                                                  int2* over, int* ctr, State* st) {
  __shared__ int h[MAXB];
  constexpr int PT = CS_TILE / 256;
  const long i0 = blockIdx.x * (long)CS_TILE + threadIdx.x;
  int key[PT], rank[PT];
#pragma unroll
  for (int q = 0; q < PT; ++q) key[q] = i0 + 256 * q < n ? map[i0 + 256 * q] : -1;
  for (int b = threadIdx.x; b < k; b += 256) h[b] = 0;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const bool live = (unsigned)key[q] < (unsigned)k;
    if (!live && i0 + 256 * q < n) atomicOr(&st->error, 2);
    rank[q] = live ? atomicAdd(&h[key[q]], 1) : 0;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < k; b += 256) {
    const int m = h[b];
    if (m) h[b] = atomicAdd(&cnt[b], m);
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const bool live = (unsigned)key[q] < (unsigned)k;
    list_member(live, key[q], live ? h[key[q]] + rank[q] : 0, (int)(i0 + 256 * q), bucket, cap, over, ctr);
  }
}

// Weighted centroid of one cluster per workgroup, its members' rho and rho * x
// (each product rounded on its own, as the reference's multiply-then-add does)
// summed in ascending grid index.
//
// The bucket holds the members in no order.  They are set as bits of a window
// of the index range (64 Ki points: a cluster of a few hundred points spans
// less on a 64^3 grid), a scan of the words' bit counts gives every member its
// rank, the values go to LDS by rank, and lanes 0..3 run the four sequential
// sums.  Up to SB_R members a thread stay in registers, their values on the
// way while the bits are counted, for up to SB_NEAR windows one after the other
// (a cluster of 256 points on a 96^3 grid may take two).  Larger clusters, and
// wider index ranges, are partitioned by window first (in 'seg', of which every such
// cluster takes as many entries as it has members), so that each member is set
// as a bit once, whatever the range; wave 0 then adds a run of members while
// the other waves look up the next run by rank.
//
// Bound by latency: two dependent loads and the chain of adds (about 9 ns
// each).  N = 262144, K = 1024: 13 us, where the stable counting sort and the
// sums that this replaces were five kernels of 40 us.
constexpr int SB_W = 2048;  // words of the window
constexpr int SB_M = 512;   // members summed at a time
constexpr int SB_R = 4;     // members a thread of the register path
constexpr int SB_NEAR = 8;  // windows of the register path
constexpr int SB_H = SB_M / 2;  // members of a run of the partitioned path
constexpr int SB_BINS = 512;    // windows partitioned at a time
static_assert(SB_W * 32 == 1 << 16, "window of an index: its bits from 16 on");

struct SumsLds {
  __attribute__((aligned(16))) unsigned bm[SB_W];
  unsigned short pre[SB_W];                            // members before a word
  int bin[SB_BINS];                                    // members by window, then where each window's end in 'seg'
  __attribute__((aligned(16))) double buf[4][SB_M + 2];  // [w, x, y, z][member], rows on different banks
  int red[4], red2[4];
  int at;
};

// v summed over the threads before this one, and over all.
__device__ inline void sums_scan(SumsLds& S, int v, int& before, int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int upto = wave_scan(v);
  if (lane == 63) S.red[wave] = upto;
  __syncthreads();
  before = upto - v;
  total = 0;
  for (int w = 0; w < 4; ++w) {
    if (w < wave) before += S.red[w];
    total += S.red[w];
  }
}

// pre of this thread's words wb .. we - 1 of the window; the window's members.
// A barrier inside, none at the end.
__device__ inline int sums_rank(SumsLds& S, int wb, int we) {
  int have = 0, pos, total;
  for (int w = wb; w < we; ++w) have += __popc(S.bm[w]);
  sums_scan(S, have, pos, total);
  for (int w = wb; w < we; ++w) {
    S.pre[w] = (unsigned short)pos;
    pos += __popc(S.bm[w]);
  }
  return total;
}

// Member of rank r of the window, as an offset into it.
__device__ inline int sums_member(const SumsLds& S, int r) {
  int w = 0;
#pragma unroll
  for (int step = SB_W / 2; step > 0; step >>= 1)
    if (S.pre[w + step] <= r) w += step;  // the last word with at most r members before it
  unsigned bits = S.bm[w], at = 0;
  int left = r - S.pre[w];
#pragma unroll
  for (int half = 16; half > 0; half >>= 1) {
    const int low = __popc(bits & ((1u << half) - 1));
    if (left >= low) {
      left -= low;
      bits >>= half;
      at += half;
    }
  }
  return 32 * w + (int)at;
}

// acc + the members seg[0 .. len) of the window at w0 in ascending order.
__device__ inline double sums_window(SumsLds& S, double acc, int w0, const int* seg, int len, const double* rho,
                                     const double* grid) {
  const int tid = threadIdx.x;
  for (int w = tid; w < SB_W / 4; w += 256) reinterpret_cast<uint4*>(S.bm)[w] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  for (int t = tid; t < len; t += 256 * 4) {
    int e[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) e[u] = t + 256 * u < len ? seg[t + 256 * u] : -1;
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (e[u] >= 0) atomicOr(&S.bm[(e[u] - w0) >> 5], 1u << (e[u] & 31));
  }
  __syncthreads();
  sums_rank(S, tid * (SB_W / 256), (tid + 1) * (SB_W / 256));
  __syncthreads();
  auto values = [&](int run) {  // of the members of a run, by waves 1 to 3
    const int h = (run & 1) * SB_H, end = min(len, (run + 1) * SB_H);
#pragma unroll 2
    for (int r = run * SB_H + tid - 64; r < end; r += 192) {
      const long e = w0 + sums_member(S, r);
      const double q = rho[e];
      double* b = &S.buf[0][h + r - run * SB_H];
      b[0] = q;
      for (int d = 0; d < 3; ++d) b[(1 + d) * (SB_M + 2)] = q * grid[e * 3 + d];
    }
  };
  const int runs = (len + SB_H - 1) / SB_H;
  if (tid >= 64) values(0);
  __syncthreads();
  for (int run = 0; run < runs; ++run) {
    if (tid < 4) acc = seq_sum(acc, &S.buf[tid][(run & 1) * SB_H], min(SB_H, len - run * SB_H));
    if (tid >= 64 && run + 1 < runs) values(run + 1);
    __syncthreads();
  }
  return acc;
}

__device__ __forceinline__ void centroid_sums_b(int* cnt, const int* bucket, int cap, const int2* over, int* ctr,
                                                     int* seg, long n, const double* rho, const double* grid, double* cen_out,
                                                     State* st, int it, int seen, int c) {
  __shared__ SumsLds S;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int* mem = bucket + (long)c * cap;
  int i[SB_R];
#pragma unroll
  for (int u = 0; u < SB_R; ++u) i[u] = tid + 256 * u < cap ? mem[tid + 256 * u] : 0;  // before the count is known
  const int m = cnt[c];
  if (st->ended <= seen || st->bad < it) return;
  const bool listed = m <= cap;
  int lo = INT_MAX, hi = INT_MAX;  // hi negated: both are minima
  double v[SB_R][4];
  const bool few = listed && m <= 256 * SB_R;
  if (few) {
#pragma unroll
    for (int u = 0; u < SB_R; ++u)
      if (tid + 256 * u < m) {
        lo = min(lo, i[u]);
        hi = min(hi, -i[u]);
        v[u][0] = rho[i[u]];
        for (int d = 0; d < 3; ++d) v[u][1 + d] = grid[i[u] * 3L + d];
      }
  }
  lo = wave_min(lo);
  hi = wave_min(hi);
  if (lane == 0) { S.red[wave] = lo; S.red2[wave] = hi; }
  for (int w = tid; w < SB_W; w += 256) S.bm[w] = 0;
  __syncthreads();
  lo = min(min(S.red[0], S.red[1]), min(S.red[2], S.red[3])) & ~31;
  hi = -min(min(S.red2[0], S.red2[1]), min(S.red2[2], S.red2[3]));
  double acc = 0.0;  // lane q < 4 of wave 0 owns accumulator q
  if (few && m > 0 && hi - lo < SB_NEAR * (SB_W * 32)) {
    for (long w0 = lo; w0 <= hi; w0 += SB_W * 32) {
      if (w0 > lo) {
        __syncthreads();
        for (int w = tid; w < SB_W; w += 256) S.bm[w] = 0;
        __syncthreads();
      }
      const int last = (int)min((long)SB_W * 32 - 1, hi - w0);
      const int per = (last >> 13) + 1, wb = tid * per;  // words a thread, all inside the window
#pragma unroll
      for (int u = 0; u < SB_R; ++u) {
        const unsigned at = (unsigned)(i[u] - w0);
        if (tid + 256 * u < m && at < SB_W * 32) atomicOr(&S.bm[at >> 5], 1u << (i[u] & 31));
      }
      __syncthreads();
      const int here = sums_rank(S, wb, wb + per);
      __syncthreads();
      for (int base = 0; base < here; base += SB_M) {
#pragma unroll
        for (int u = 0; u < SB_R; ++u) {
          const unsigned at = (unsigned)(i[u] - w0);
          if (tid + 256 * u < m && at < SB_W * 32) {
            const int w = at >> 5;
            const int r = S.pre[w] + __popc(S.bm[w] & ((1u << (i[u] & 31)) - 1)) - base;
            if (r >= 0 && r < SB_M) {
              S.buf[0][r] = v[u][0];
              for (int d = 0; d < 3; ++d) S.buf[1 + d][r] = v[u][0] * v[u][1 + d];
            }
          }
        }
        __syncthreads();
        if (tid < 4) acc = seq_sum(acc, S.buf[tid], min(SB_M, here - base));
        if (base + SB_M < here) __syncthreads();
      }
    }
  } else if (m > 0) {
    // every member: f(grid index), eight loads in flight
    const int nb = min(m, cap), no = listed ? 0 : ctr[it & 1];
    auto members = [&](auto f) {
      for (int t = tid; t < nb; t += 256 * 8) {
        int e[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) e[u] = t + 256 * u < nb ? mem[t + 256 * u] : -1;
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (e[u] >= 0) f(e[u]);
      }
      for (int t = tid; t < no; t += 256 * 8) {
        int2 e[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) e[u] = t + 256 * u < no ? over[t + 256 * u] : make_int2(-1, 0);
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (e[u].x == c) f(e[u].y);
      }
    };
    if (tid == 0) S.at = atomicAdd(&ctr[2 + (it & 1)], m);
    __syncthreads();
    int base = S.at;
    for (long r0 = 0; r0 < n; r0 += SB_BINS * (SB_W * 32L)) {
      for (int q = tid; q < SB_BINS; q += 256) S.bin[q] = 0;
      __syncthreads();
      members([&](int e) {
        const long q = (e - r0) >> 16;
        if (e >= r0 && q < SB_BINS) atomicAdd(&S.bin[q], 1);
      });
      __syncthreads();
      const int h0 = S.bin[2 * tid], h1 = S.bin[2 * tid + 1];
      int before, total;
      sums_scan(S, h0 + h1, before, total);
      S.bin[2 * tid] = base + before;
      S.bin[2 * tid + 1] = base + before + h0;
      __syncthreads();
      members([&](int e) {
        const long q = (e - r0) >> 16;
        if (e >= r0 && q < SB_BINS) seg[atomicAdd(&S.bin[q], 1)] = e;
      });
      __syncthreads();
      const int windows = (int)min((long)SB_BINS, (n - r0 + SB_W * 32 - 1) / (SB_W * 32));
      for (int q = 0; q < windows; ++q) {
        const int end = S.bin[q];
        if (end > base) acc = sums_window(S, acc, (int)r0 + q * (SB_W * 32), seg + base, end - base, rho, grid);
        base = end;
      }
      __syncthreads();
    }
  }
  if (tid >= 64) return;
  const double w = __shfl(acc, 0);
  if (lane == 0) {
    cnt[c] = 0;  // empty for the next assignment
    if (w < 1e-8) atomicMin(&st->bad, it);
  }
  if (lane >= 1 && lane < 4) cen_out[c * 3 + lane - 1] = acc / w;
}
__global__ __launch_bounds__(256) void centroid_sums(int* cnt, const int* bucket, int cap, const int2* over, int* ctr,
                                                     int* seg, long n, const double* rho, const double* grid,
                                                     double* cen_out, State* st, int it, int seen) {
  centroid_sums_b(cnt, bucket, cap, over, ctr, seg, n, rho, grid, cen_out, st, it, seen, (int)blockIdx.x);
}

// normed_difference(new, cur) with the reference's sequential sum, % changed,
// and the loop control of KMeansSolver::kernel (kmeans.cpp:233-257).  chg: the
// iteration's CHG partial change counts.  Where the threshold cannot stop the
// loop (Layout::defer) every iteration's is run after the loop, side by side.
__device__ __forceinline__ void diff_control_b(const double* nxt, const double* cur, int k, long n,
                                                     double threshold, int it, int max_it, int nxt_buf,
                                                     State* st, int* chg, double* diffs, double* pcts,
                                                     bool defer) {
  if (!defer && st->ended < it) return;
  extern __shared__ __attribute__((aligned(16))) double terms[];
  __shared__ double red[4][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int len = 3 * k;
  const int bad = st->bad;
  if (bad <= it) {
    if (bad == it && tid == 0) {
      st->error = 1;
      st->iters = it + 1;
      if (!defer) st->ended = it;
    }
    return;
  }
  double mxa = -DBL_MAX, mna = DBL_MAX, mxb = -DBL_MAX, mnb = DBL_MAX;
  for (int i = tid; i < len; i += 1024) {
    mxa = fmax(mxa, nxt[i]); mna = fmin(mna, nxt[i]);
    mxb = fmax(mxb, cur[i]); mnb = fmin(mnb, cur[i]);
  }
  mxa = -wave_min(-mxa); mna = wave_min(mna); mxb = -wave_min(-mxb); mnb = wave_min(mnb);
  if (lane == 0) { red[0][wave] = mxa; red[1][wave] = mna; red[2][wave] = mxb; red[3][wave] = mnb; }
  __syncthreads();
  mxa = red[0][0]; mna = red[1][0]; mxb = red[2][0]; mnb = red[3][0];
  for (int w = 1; w < 16; ++w) {
    mxa = fmax(mxa, red[0][w]); mna = fmin(mna, red[1][w]);
    mxb = fmax(mxb, red[2][w]); mnb = fmin(mnb, red[3][w]);
  }
  const double scale = fmax(fabs(mxa), fabs(mna)) + fmax(fabs(mxb), fabs(mnb));
  for (int i = tid; i < len; i += 1024) {
    const double t = (nxt[i] - cur[i]) / scale;
    terms[i] = t * t;
  }
  __syncthreads();
  if (wave > 0) return;
  const int changed = wave_sum(lane < CHG ? chg[lane] : 0);
  if (!defer && lane < CHG) chg[lane] = 0;
  if (lane == 0) {
    const double diff = scale * sqrt(seq_sum(0.0, terms, len));  // the reference's order
    const double pct = 100 * ((double)changed) / (double)n;
    diffs[it] = diff;
    pcts[it] = pct;
    if (!defer || it == max_it - 1) st->iters = it + 1;
    if (!defer || it == max_it - 1 || bad == it + 1) st->last_diff = diff;
    if (diff < threshold) {
      st->ended = it;
      st->mode = MODE_FINAL;
      st->final_buf = nxt_buf;
    } else if (it == max_it - 1) {
      st->mode = (diff > threshold) ? MODE_LATEST : MODE_ZEROS;
    }
  }
}
__global__ __launch_bounds__(1024) void diff_control(const double* nxt, const double* cur, int k, long n,
                                                     double threshold, int it, int max_it, int nxt_buf,
                                                     State* st, int* chg, double* diffs, double* pcts) {
  diff_control_b(nxt, cur, k, n, threshold, it, max_it, nxt_buf, st, chg, diffs, pcts, false);
}
// all iterations of a run that kept every iteration's centroids
__global__ __launch_bounds__(1024) void diff_control_all(const double* cen, int k, long n, double threshold, int max_it,
                                                         State* st, int* chg, double* diffs, double* pcts) {
  const int it = (int)blockIdx.x;
  const long cs = 3L * k;
  diff_control_b(cen + (it + 1) * cs, cen + it * cs, k, n, threshold, it, max_it, it + 1, st, chg + it * CHG, diffs,
                 pcts, true);
}

// ------------------------------------------------------------------ map_to_grid

// Nearest grid point per centroid (lexicographic distance/index minimum over
// the grid tiles the bounds cannot exclude).  beside: the loop control runs
// after the loop, beside this kernel: a vanished weight is known from the sums
// alone, and 'mode', which it may be writing, is not read (all of a workgroup's
// waves take one way; sort_indices zeroes the points of MODE_ZEROS).  Else it
// has ended, and only its verdict counts (the iteration that a converged loop
// had started may have set 'bad').
__device__ __forceinline__ void map_to_grid_b(const double* sx, const double* sy, const double* sz,
                                                   const int* perm, long n, const double* boxes, int ntiles,
                                                   const double* cen3, long cstride, int latest_buf,
                                                   const State* st, bool beside, int* out, int bid) {
  const int c = bid;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int mode = st && !beside ? st->mode : MODE_LATEST;
  if (mode == MODE_ZEROS || (st && (beside ? st->bad != INT_MAX : st->error != 0))) {
    if (tid == 0) out[c] = 0;
    return;
  }
  const int buf = (mode == MODE_FINAL) ? st->final_buf : latest_buf;
  const double* cen = cen3 + buf * cstride;
  const double cx = cen[c * 3], cy = cen[c * 3 + 1], cz = cen[c * 3 + 2];
  __shared__ double redd[4];
  __shared__ int redi[4];
  __shared__ int tl[MAXB];
  double u = DBL_MAX;
  for (int t = tid; t < ntiles; t += 256) u = fmin(u, ub2_box(cx, cy, cz, boxes + (long)t * 6));
  u = wave_min(u);
  if (lane == 0) redd[wave] = u;
  __syncthreads();
  u = fmin(fmin(redd[0], redd[1]), fmin(redd[2], redd[3]));
  const double thr = u * PRUNE;
  double bd2 = DBL_MAX, bs = DBL_MAX;
  int bi = INT_MAX;
  __shared__ int cntw;
  // candidate tiles, collected in windows of MAXB
  for (int t0 = 0; t0 < ntiles; t0 += MAXB) {
    const int tend = min(ntiles, t0 + MAXB);
    if (tid == 0) cntw = 0;
    __syncthreads();
    for (int t = t0 + tid; t < tend; t += 256)
      if (lb2_box(cx, cy, cz, boxes + (long)t * 6) <= thr) tl[atomicAdd(&cntw, 1)] = t;
    __syncthreads();
    const int nt = cntw;
    for (int q = 0; q < nt; ++q) {
      const long p = (long)tl[q] * TP + tid;
      if (p < n) consider_any(dist2(sx[p], sy[p], sz[p], cx, cy, cz), perm[p], bd2, bs, bi);
    }
    __syncthreads();
  }
  // lexicographic reduction of (bs, bi)
  for (int o = 32; o > 0; o >>= 1) {
    const double os = __shfl_xor(bs, o);
    const int oi = __shfl_xor(bi, o);
    if (os < bs || (os == bs && oi < bi)) { bs = os; bi = oi; }
  }
  if (lane == 0) { redd[wave] = bs; redi[wave] = bi; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w)
      if (redd[w] < bs || (redd[w] == bs && redi[w] < bi)) { bs = redd[w]; bi = redi[w]; }
    // redd[0]/redi[0] already folded through bs/bi of wave 0
    out[c] = bi;
  }
}
__global__ __launch_bounds__(256) void map_to_grid(const double* sx, const double* sy, const double* sz,
                                                   const int* perm, long n, const double* boxes, int ntiles,
                                                   const double* cen3, long cstride, int latest_buf,
                                                   const State* st, bool beside, int* out) {
  map_to_grid_b(sx, sy, sz, perm, n, boxes, ntiles, cen3, cstride, latest_buf, st, beside, out, (int)blockIdx.x);
}

// Sort the k indices ascending (bitonic in LDS) and count adjacent repeats; a
// run that ended without points (MODE_ZEROS, an error) has zeros.
__device__ __forceinline__ void sort_indices_b(int* idx, int k, State* st) {
  __shared__ int s[MAXB];
  int p2 = 1;
  while (p2 < k) p2 <<= 1;
  const bool none = st && (st->mode == MODE_ZEROS || st->error != 0);
  for (int i = threadIdx.x; i < p2; i += 1024) s[i] = i >= k ? INT_MAX : (none ? 0 : idx[i]);
  __syncthreads();
  for (int size = 2; size <= p2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < p2; i += 1024) {
        const int j = i ^ stride;
        if (j > i) {
          const bool up = (i & size) == 0;
          const int a = s[i], b = s[j];
          if ((a > b) == up) { s[i] = b; s[j] = a; }
        }
      }
      __syncthreads();
    }
  }
  int d = 0;
  for (int i = threadIdx.x; i < k; i += 1024) {
    idx[i] = s[i];
    if (i + 1 < k && s[i] == s[i + 1]) ++d;
  }
  d = wave_sum(d);
  if ((threadIdx.x & 63) == 0 && d && st) atomicAdd(&st->dups, d);
}
__global__ __launch_bounds__(1024) void sort_indices(int* idx, int k, State* st) {
  sort_indices_b(idx, k, st);
}

}  // namespace km
}  // namespace thc

// ====================================================================== host

namespace thc {
namespace km {

// final assignment (kept in tile order) and centroids
__global__ void copy_final(const int* map0, const int* map1, const int* perm, long n, const double* cen3, int k,
                           int latest_buf, const State* st, int* map_out, double* cen_out) {
  const int iters = st->iters;
  const int mbuf = iters > 0 ? (iters - 1) & 1 : 0;
  const int cbuf = st->mode == MODE_FINAL ? st->final_buf : latest_buf;
  const int* m = mbuf ? map1 : map0;
  const double* c = cen3 + cbuf * 3L * k;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += 256L * gridDim.x) {
    if (map_out) map_out[perm[i]] = m[i];
    if (cen_out && i < 3L * k) cen_out[i] = c[i];
  }
  if (cen_out && n < 3L * k)
    for (long i = n + blockIdx.x * 256L + threadIdx.x; i < 3L * k; i += 256L * gridDim.x) cen_out[i] = c[i];
}

// f with the assignment's centroids a thread for k clusters, as a constant
template <class F>
static void with_cpt(int k, F f) {
  if (k <= 256) f(std::integral_constant<int, 1>{});
  else if (k <= 1024) f(std::integral_constant<int, 4>{});
  else if (k <= 2048) f(std::integral_constant<int, 8>{});
  else f(std::integral_constant<int, MAXB / 256>{});
}

struct Layout {
  long n;
  int k, max_it;
  int cells, nbins_sp, nbits_sp;
  int ntiles, ncs, nbb;
  int cap;      // members a cluster's bucket holds
  int defer;    // the threshold cannot stop the loop: every iteration's centroids are kept, the differences come last
  int ncen;     // centroid buffers
  int nchg;     // iterations' change counts kept
};

static int bits_for(int nb) {
  int b = 1;
  while ((1 << b) < nb) ++b;
  return b;
}

// Members a cluster's bucket holds: eight times the average (the largest
// clusters of filled 64^3 cells reach four times); those of larger clusters, as
// vacuum around a molecule or slab gives, share one list.
static int bucket_cap(long n, int k) { return (int)std::min<long>(n, std::max<long>(256, 8 * ((n + k - 1) / k))); }

// A normed difference is never negative, so a negative threshold never stops
// the loop, and nothing in it waits for the differences.
constexpr size_t DEFER_BYTES = size_t(64) << 20;  // kept centroids of one run
static bool can_defer(int k, int max_it, double threshold) {
  const size_t each = sizeof(double) * 3 * (size_t)k + sizeof(int) * CHG;
  return !(threshold >= 0.0) && each * ((size_t)max_it + 1) <= DEFER_BYTES;
}

static Layout plan(long n, int k, int max_it, bool defer) {
  Layout L;
  L.n = n; L.k = k; L.max_it = max_it;
  int cells = 1;
  while (cells < 16 && (long)(2 * cells) * (2 * cells) * (2 * cells) * 64 <= n) cells *= 2;
  L.cells = cells;
  L.nbins_sp = cells * cells * cells;
  L.nbits_sp = bits_for(L.nbins_sp);
  L.ntiles = ceil_div(n, TP);
  L.ncs = ceil_div(n, CS_TILE);
  L.nbb = (int)std::min<long>(256, (n + 255) / 256);
  L.cap = bucket_cap(n, k);
  L.defer = defer;
  L.ncen = defer ? max_it + 1 : 3;
  L.nchg = defer ? max_it : 4;
  return L;
}

struct Bufs {
  double *part, *sx, *sy, *sz, *boxes, *wboxes, *cen, *diffs, *pcts;  // cen: L.ncen centroid buffers
  int *keys, *perm, *map[2], *tc, *total, *start, *idx0;     // map: in tile order
  int *cnt, *bucket, *ctr, *seg, *chg;
  int2* over;
  State* st;
};

static size_t bytes_for(const Layout& L, bool full) {
  const long n = L.n;
  const int nb = L.nbins_sp;
  size_t b = 0;
  b += carve_bytes<double>(L.nbb * 6);
  b += 3 * carve_bytes<double>(n) + carve_bytes<double>((size_t)L.ntiles * 6) + carve_bytes<double>((size_t)L.ntiles * 24);
  b += 2 * carve_bytes<int>(n);                       // keys, perm
  b += carve_bytes<int>((size_t)L.ncs * nb) + 2 * carve_bytes<int>(nb);
  b += carve_bytes<State>(1);
  if (full) {
    b += carve_bytes<double>(3L * L.k * L.ncen) + 2 * carve_bytes<double>(std::max(1, L.max_it));
    b += 2 * carve_bytes<int>(n) + carve_bytes<int>(L.k);
    b += carve_bytes<int>(L.k) + carve_bytes<int>((size_t)L.k * L.cap) + carve_bytes<int>((size_t)L.nchg * CHG);
    b += carve_bytes<int>(4) + carve_bytes<int>(n) + carve_bytes<int2>(n);
  }
  return b;
}

static bool carve(Arena& a, const Layout& L, Bufs& b, bool full) {
  const long n = L.n;
  const int nb = L.nbins_sp;
  b = Bufs{};
  b.part = a.take<double>(L.nbb * 6);
  b.sx = a.take<double>(n);
  b.sy = a.take<double>(n);
  b.sz = a.take<double>(n);
  b.boxes = a.take<double>((size_t)L.ntiles * 6);
  b.wboxes = a.take<double>((size_t)L.ntiles * 24);
  b.keys = a.take<int>(n);
  b.perm = a.take<int>(n);
  b.tc = a.take<int>((size_t)L.ncs * nb);
  b.total = a.take<int>(nb);
  b.start = a.take<int>(nb);
  b.st = a.take<State>(1);
  bool ok = b.part && b.sx && b.sy && b.sz && b.boxes && b.wboxes && b.keys && b.perm && b.tc && b.total && b.start && b.st;
  if (full) {
    b.cen = a.take<double>(3L * L.k * L.ncen);
    b.diffs = a.take<double>(std::max(1, L.max_it));
    b.pcts = a.take<double>(std::max(1, L.max_it));
    b.map[0] = a.take<int>(n);
    b.map[1] = a.take<int>(n);
    b.idx0 = a.take<int>(L.k);
    b.cnt = a.take<int>(L.k);
    b.bucket = a.take<int>((size_t)L.k * L.cap);
    b.chg = a.take<int>((size_t)L.nchg * CHG);
    b.ctr = a.take<int>(4);
    b.seg = a.take<int>(n);
    b.over = a.take<int2>(n);
    ok = ok && b.cen && b.diffs && b.pcts && b.map[0] && b.map[1] && b.idx0 && b.cnt && b.bucket && b.chg && b.ctr &&
         b.seg && b.over;
  }
  return ok;
}

// Spatially sorted copy of the grid (a stable counting sort by Morton cell)
// and tile boxes.
static void enqueue_setup(const Layout& L, const Bufs& b, const double* grid, hipStream_t s) {
  hipLaunchKernelGGL(bbox_partial, dim3(L.nbb), dim3(256), 0, s, grid, L.n, b.part);
  hipLaunchKernelGGL(morton_keys, dim3(ceil_div(L.n, 256)), dim3(256), 0, s, grid, L.n, b.part, L.nbb, L.cells, b.keys);
  hipLaunchKernelGGL(cs_hist, dim3(L.ncs), dim3(256), 0, s, b.keys, L.n, L.nbins_sp, b.tc);
  hipLaunchKernelGGL(cs_colscan, dim3(ceil_div(L.nbins_sp, 64)), dim3(64 * CS_SCAN_W), 0, s, b.tc, L.ncs, L.nbins_sp,
                     b.total);
  hipLaunchKernelGGL(cs_totscan, dim3(1), dim3(1024), 0, s, b.total, L.nbins_sp, b.start);
  hipLaunchKernelGGL(cs_scatter, dim3(L.ncs), dim3(256), 0, s, b.keys, L.n, L.nbins_sp, L.nbits_sp, b.tc, b.start,
                     b.perm);
  hipLaunchKernelGGL(sorted_tiles, dim3(L.ntiles), dim3(256), 0, s, grid, b.perm, L.n, b.sx, b.sy, b.sz, b.boxes,
                     b.wboxes);
}

// centroid buffer iteration 'it' reads; it writes that of it + 1
__host__ __device__ inline int cen_buf(const Layout& L, int it) { return L.defer ? it : it % 3; }
// and its change counts (iteration it + 4 starts after the loop control of it,
// which clears them)
__host__ __device__ inline long chg_at(const Layout& L, int it) { return (long)(L.defer ? it : it & 3) * CHG; }

// An iteration is two kernels, the assignment and the centroid sums.
//
// Where the threshold cannot stop the loop (L.defer) it keeps every
// iteration's centroids, and the normed differences -- chains of 3 k
// sequential adds -- are formed after it, one workgroup per iteration, beside
// map_to_grid on the second stream.
//
// Otherwise the loop control of iteration it (diff_control: the difference,
// the stop test) runs on the second stream beside iteration it + 1, which does
// not need its result: if iteration it stops the loop, iteration it + 1
// (already started) only writes buffers the final state does not use, and
// iteration it + 2 waits for it and returns at once.  Iteration it + 1 runs to
// its end even if the stop comes while it runs: its workgroups go only by
// controls that had ended before they started ('seen'), so the waves of one
// never part at a flag that changes under them.  Hence three centroid
// buffers (iteration it reads it % 3, writes (it+1) % 3, and diff_control(it)
// still reads both while iteration it + 1 writes (it+2) % 3).  With sa == s
// the same code runs in order on one stream.
static int enqueue_kmeans(const Layout& L, const Bufs& b, const double* grid, const double* rho, double threshold,
                          int* interp_idx, int* map_out, double* cen_out, hipStream_t s, hipStream_t sa,
                          const hipEvent_t kev[3]) {
  const long cs = 3L * L.k;
  const bool two = sa != s;
  hipLaunchKernelGGL(init_run, dim3(ceil_div(L.k, 256)), dim3(256), 0, s, grid, b.idx0, L.k, b.cen, b.cnt, b.ctr, b.chg,
                     L.nchg * CHG, b.st);
  enqueue_setup(L, b, grid, s);
  const size_t dyn = (size_t)3 * L.k * sizeof(double);
  for (int it = 0; it < L.max_it; ++it) {
    const int cur = cen_buf(L, it), nxt = cen_buf(L, it + 1), par = it & 1;
    const int seen = it - (two ? 2 : 1);  // the latest loop control this iteration starts after
    int* mnew = b.map[par];
    const int* mold = it == 0 ? nullptr : b.map[par ^ 1];
    if (!L.defer && two && it >= 2) THC_HIP(hipStreamWaitEvent(s, kev[1 + par], 0));  // diff_control(it - 2)
    with_cpt(L.k, [&](auto cpt) {
      hipLaunchKernelGGL(assign<cpt.value>, dim3(L.ntiles), dim3(256), 0, s, b.sx, b.sy, b.sz, b.perm, L.n, b.boxes,
                         b.wboxes, b.cen + cur * cs, L.k, mnew, mold, b.cnt, b.bucket, L.cap, b.over, b.ctr,
                         b.chg + chg_at(L, it), b.st, it, seen);
    });
    hipLaunchKernelGGL(centroid_sums, dim3(L.k), dim3(256), 0, s, b.cnt, b.bucket, L.cap, b.over, b.ctr, b.seg,
                       L.n, rho, grid, b.cen + nxt * cs, b.st, it, seen);
    if (L.defer) continue;
    if (two) {
      THC_HIP(hipEventRecord(kev[0], s));
      THC_HIP(hipStreamWaitEvent(sa, kev[0], 0));
    }
    hipLaunchKernelGGL(diff_control, dim3(1), dim3(1024), dyn, sa, b.cen + nxt * cs, b.cen + cur * cs, L.k, L.n,
                       threshold, it, L.max_it, nxt, b.st, b.chg + chg_at(L, it), b.diffs, b.pcts);
    if (two) THC_HIP(hipEventRecord(kev[1 + par], sa));
  }
  const int last = 1 + ((L.max_it - 1) & 1);
  if (L.defer) {
    if (two) {
      THC_HIP(hipEventRecord(kev[0], s));
      THC_HIP(hipStreamWaitEvent(sa, kev[0], 0));
    }
    hipLaunchKernelGGL(diff_control_all, dim3(L.max_it), dim3(1024), dyn, sa, b.cen, L.k, L.n, threshold, L.max_it,
                       b.st, b.chg, b.diffs, b.pcts);
    if (two) THC_HIP(hipEventRecord(kev[last], sa));
  }
  // the last loop control: map_to_grid goes by its verdict where there is one
  if (two && !L.defer) THC_HIP(hipStreamWaitEvent(s, kev[last], 0));
  const int latest = cen_buf(L, L.max_it);
  hipLaunchKernelGGL(map_to_grid, dim3(L.k), dim3(256), 0, s, b.sx, b.sy, b.sz, b.perm, L.n, b.boxes, L.ntiles,
                     b.cen, cs, latest, b.st, L.defer != 0, interp_idx);
  if (two && L.defer) THC_HIP(hipStreamWaitEvent(s, kev[last], 0));
  hipLaunchKernelGGL(sort_indices, dim3(1), dim3(1024), 0, s, interp_idx, L.k, b.st);
  if (map_out || cen_out)
    hipLaunchKernelGGL(copy_final, dim3(256), dim3(256), 0, s, b.map[0], b.map[1], b.perm, L.n, b.cen, L.k, latest,
                       b.st, map_out, cen_out);
  THC_HIP(hipGetLastError());
  return THC_OK;
}

// ------------------------------------------------------------------ batches
//
// A batch runs the k-means of many systems together: every launch below
// covers one step (setup, assignment, centroid sums, loop control, map to
// grid) of all the systems, so a 20-iteration batch of 32 systems is about 50
// launches instead of 32 times that.  Each workgroup finds its system in
// a prefix table of per-system block counts and runs the same device code as
// the single-system kernels with that system's sizes and buffers, so every
// system's result is bit-identical to its own thc_kmeans.

struct Job {
  Layout L;
  Bufs b;
  const double* grid;
  const double* rho;
  double threshold;
  int* interp_idx;
};

// block-count tables, one row of nj + 1 prefix sums per kind
enum { JK_NBB, JK_N256, JK_NCS, JK_COLSP, JK_TILES, JK_K256, JK_K, JK_COUNT };

inline int job_blocks(const Layout& L, int kind) {
  switch (kind) {
    case JK_NBB: return L.nbb;
    case JK_N256: return (int)ceil_div(L.n, 256);
    case JK_NCS: return L.ncs;
    case JK_COLSP: return ceil_div(L.nbins_sp, 64);
    case JK_TILES: return L.ntiles;
    case JK_K256: return ceil_div(L.k, 256);
    default: return L.k;
  }
}

// system of workgroup b: off[j] <= b < off[j + 1]
__device__ inline int job_of(const int* off, int nj, int b) {
  int lo = 0, hi = nj;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}

#define KM_JOB(OFF)                                 \
  const int j_ = job_of(OFF, nj, (int)blockIdx.x);  \
  const Job& q = jobs[j_];                          \
  const int bid = (int)blockIdx.x - OFF[j_], nblk = OFF[j_ + 1] - OFF[j_];

__global__ __launch_bounds__(256) void init_run_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  init_run_b(q.grid, q.b.idx0, q.L.k, q.b.cen, q.b.cnt, q.b.ctr, q.b.chg, q.L.nchg * CHG, q.b.st, bid, nblk);
}

__global__ __launch_bounds__(256) void bbox_partial_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  bbox_partial_b(q.grid, q.L.n, q.b.part, bid, nblk);
}

__global__ __launch_bounds__(256) void morton_keys_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  (void)nblk;
  morton_keys_b(q.grid, q.L.n, q.b.part, q.L.nbb, q.L.cells, q.b.keys, bid);
}

__global__ __launch_bounds__(256) void cs_hist_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  cs_hist_b(q.b.keys, q.L.n, q.L.nbins_sp, q.b.tc, bid, nblk);
}

__global__ __launch_bounds__(64 * CS_SCAN_W) void cs_colscan_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  cs_colscan_b(q.b.tc, q.L.ncs, q.L.nbins_sp, q.b.total, bid, nblk);
}

__global__ __launch_bounds__(1024) void cs_totscan_m(const Job* jobs) {
  const Job& q = jobs[blockIdx.x];
  cs_totscan_b(q.b.total, q.L.nbins_sp, q.b.start, 0, 1);
}

__global__ __launch_bounds__(256) void cs_scatter_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  cs_scatter_b(q.b.keys, q.L.n, q.L.nbins_sp, q.L.nbits_sp, q.b.tc, q.b.start, q.b.perm, bid, nblk);
}

__global__ __launch_bounds__(256) void sorted_tiles_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  (void)nblk;
  sorted_tiles_b(q.grid, q.b.perm, q.L.n, q.b.sx, q.b.sy, q.b.sz, q.b.boxes, q.b.wboxes, bid);
}

__device__ inline double* job_cen(const Job& q, int it) { return q.b.cen + cen_buf(q.L, it) * 3L * q.L.k; }

template <int CPT>
__global__ __launch_bounds__(256) void assign_m(const Job* jobs, const int* off, int nj, int it) {
  KM_JOB(off)
  (void)nblk;
  if (it >= q.L.max_it) return;
  const int par = it & 1;
  assign_b<CPT>(q.b.sx, q.b.sy, q.b.sz, q.b.perm, q.L.n, q.b.boxes, q.b.wboxes, job_cen(q, it), q.L.k, q.b.map[par],
           it == 0 ? nullptr : q.b.map[par ^ 1], q.b.cnt, q.b.bucket, q.L.cap, q.b.over, q.b.ctr,
           q.b.chg + chg_at(q.L, it), q.b.st, it, it - 1, bid);
}

__global__ __launch_bounds__(256) void centroid_sums_m(const Job* jobs, const int* off, int nj, int it) {
  KM_JOB(off)
  (void)nblk;
  if (it >= q.L.max_it) return;
  centroid_sums_b(q.b.cnt, q.b.bucket, q.L.cap, q.b.over, q.b.ctr, q.b.seg, q.L.n, q.rho, q.grid, job_cen(q, it + 1),
                  q.b.st, it, it - 1, bid);
}

// loop control of iteration it0 + blockIdx.y
__global__ __launch_bounds__(1024) void diff_control_m(const Job* jobs, int it0) {
  const Job& q = jobs[blockIdx.x];
  const int it = it0 + (int)blockIdx.y;
  if (it >= q.L.max_it) return;
  diff_control_b(job_cen(q, it + 1), job_cen(q, it), q.L.k, q.L.n, q.threshold, it, q.L.max_it,
                 cen_buf(q.L, it + 1), q.b.st, q.b.chg + chg_at(q.L, it), q.b.diffs, q.b.pcts, q.L.defer);
}

__global__ __launch_bounds__(256) void map_to_grid_m(const Job* jobs, const int* off, int nj) {
  KM_JOB(off)
  (void)nblk;
  map_to_grid_b(q.b.sx, q.b.sy, q.b.sz, q.b.perm, q.L.n, q.b.boxes, q.L.ntiles, q.b.cen, 3L * q.L.k,
                cen_buf(q.L, q.L.max_it), q.b.st, q.L.defer != 0, q.interp_idx, bid);
}

__global__ __launch_bounds__(1024) void sort_indices_m(const Job* jobs) {
  const Job& q = jobs[blockIdx.x];
  sort_indices_b(q.interp_idx, q.L.k, q.b.st);
}

// every system's State, diffs and pcts into one block for a single copy back:
// system j at out + j * stride bytes
constexpr long STATE_SLOT = (sizeof(State) + 63) / 64 * 64;  // State, then diffs and pcts

__global__ void collect_m(const Job* jobs, char* out, long stride, int max_it) {
  const Job& q = jobs[blockIdx.x];
  char* o = out + blockIdx.x * stride;
  const int t = threadIdx.x;
  if (t == 0) *reinterpret_cast<State*>(o) = *q.b.st;
  double* d = reinterpret_cast<double*>(o + STATE_SLOT);
  for (int i = t; i < max_it; i += blockDim.x) {
    d[i] = i < q.L.max_it ? q.b.diffs[i] : 0.0;
    d[max_it + i] = i < q.L.max_it ? q.b.pcts[i] : 0.0;
  }
}

#undef KM_JOB

}  // namespace km

static std::atomic<int> km_attrs_done{0};  // batched calls run two k-means at once
static int km_set_attrs() {
  if (km_attrs_done) return THC_OK;
  for (const void* f : {(const void*)km::diff_control, (const void*)km::diff_control_all,
                        (const void*)km::diff_control_m})
    THC_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 3 * km::MAXB * (int)sizeof(double)));
  km_attrs_done = 1;
  return THC_OK;
}

int kmeans_run(thc_ctx* ctx, const double* grid, const double* rho, long n, int k, int max_it, double threshold,
               const int* host_init_idx, int* interp_idx, int* grid_map_out, double* centroids_out,
               thc_kmeans_stats* stats) {
  using namespace km;
  if (!ctx || !grid || !rho || !interp_idx || !host_init_idx) return THC_ERR_ARG;
  if (n < 1 || k < 1 || k > n || max_it < 1 || n > 0x7fffffffL) return THC_ERR_ARG;
  if (k > MAXB) return THC_ERR_UNSUPPORTED;
  for (int j = 0; j < k; ++j)
    if (host_init_idx[j] < 0 || host_init_idx[j] >= n) {
      set_last_error("a starting index lies outside [0, n)", __FILE__, __LINE__);
      return THC_ERR_ARG;
    }
  THC_HIP(hipSetDevice(ctx->device));
  THC_TRY(km_set_attrs());
  const Layout L = plan(n, k, max_it, can_defer(k, max_it, threshold));
  const size_t need = bytes_for(L, true);
  if (need > ctx->kmws.cap) {
    if (ctx->kmgraph) ctx->kmgraph->reset();
    THC_TRY(ctx->kmws.reserve(need));
  }
  ctx->kmws.reset();
  Bufs b;
  if (!carve(ctx->kmws, L, b, true)) return THC_ERR_NO_MEMORY;
  hipStream_t s = ctx->stream;
  THC_TRY(ensure_pinned(ctx, sizeof(int) * k + sizeof(State) + 2 * sizeof(double) * max_it + 64));
  int* hidx = reinterpret_cast<int*>(ctx->pinned);
  std::copy(host_init_idx, host_init_idx + k, hidx);
  THC_HIP(hipEventRecord(ctx->ev[0], s));
  THC_HIP(hipMemcpyAsync(b.idx0, hidx, sizeof(int) * k, hipMemcpyHostToDevice, s));
  if (ctx->use_graphs) {
    if (!ctx->kmgraph) ctx->kmgraph = new KmGraphCache();
    KmGraphCache& gc = *ctx->kmgraph;
    const void* key[5] = {grid, rho, interp_idx, grid_map_out, centroids_out};
    bool hit = gc.exec && gc.n == n && gc.k == k && gc.max_it == max_it && gc.threshold == threshold &&
               gc.base == ctx->kmws.base && gc.overlap == ctx->km_overlap;
    for (int q = 0; q < 5 && hit; ++q) hit = gc.key_ptr[q] == key[q];
    if (!hit) {
      gc.reset();
      THC_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      const int est = enqueue_kmeans(L, b, grid, rho, threshold, interp_idx, grid_map_out, centroids_out, s,
                                     ctx->km_overlap ? ctx->aux : s, ctx->kev);
      hipError_t e = hipStreamEndCapture(s, &gc.graph);
      THC_TRY(est);
      THC_HIP(e);
      THC_HIP(hipGraphInstantiate(&gc.exec, gc.graph, nullptr, nullptr, 0));
      for (int q = 0; q < 5; ++q) gc.key_ptr[q] = key[q];
      gc.n = n; gc.k = k; gc.max_it = max_it; gc.threshold = threshold; gc.base = ctx->kmws.base;
      gc.overlap = ctx->km_overlap;
    }
    THC_HIP(hipGraphLaunch(gc.exec, s));
  } else {
    THC_TRY(enqueue_kmeans(L, b, grid, rho, threshold, interp_idx, grid_map_out, centroids_out, s,
                           ctx->km_overlap ? ctx->aux : s, ctx->kev));
  }
  char* hp = reinterpret_cast<char*>(ctx->pinned);
  State* hst = reinterpret_cast<State*>(hp + align_up(sizeof(int) * k, 64));
  double* hd = reinterpret_cast<double*>(reinterpret_cast<char*>(hst) + align_up(sizeof(State), 64));
  double* hpct = hd + max_it;
  THC_HIP(hipMemcpyAsync(hst, b.st, sizeof(State), hipMemcpyDeviceToHost, s));
  THC_HIP(hipMemcpyAsync(hd, b.diffs, sizeof(double) * max_it, hipMemcpyDeviceToHost, s));
  THC_HIP(hipMemcpyAsync(hpct, b.pcts, sizeof(double) * max_it, hipMemcpyDeviceToHost, s));
  THC_HIP(hipEventRecord(ctx->ev[1], s));
  THC_HIP(hipStreamSynchronize(s));
  if (stats) {
    stats->iterations = hst->iters;
    stats->converged = hst->mode == MODE_FINAL;
    stats->duplicates = hst->dups;
    stats->interp_zeroed = hst->mode == MODE_ZEROS;
    stats->last_diff = hst->last_diff;
    if (stats->diffs) std::copy(hd, hd + hst->iters, stats->diffs);
    if (stats->pcts) std::copy(hpct, hpct + hst->iters, stats->pcts);
    float ms = 0;
    THC_HIP(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
    stats->elapsed_ms = ms;
  }
  if (hst->error) return THC_ERR_EMPTY_CLUSTER;
  if (hst->dups) return THC_WARN_DUPLICATE_INDICES;
  return THC_OK;
}


extern "C" int thc_seed_indices_impl(long n, int k, unsigned int seed, int* out);

int kmeans_run_many(thc_ctx* ctx, int nj, const KmSpec* spec, int* status, thc_kmeans_stats* stats) {
  using namespace km;
  if (!ctx || nj < 0 || (nj > 0 && (!spec || !status))) return THC_ERR_ARG;
  if (nj == 0) return THC_OK;
  THC_HIP(hipSetDevice(ctx->device));
  THC_TRY(km_set_attrs());
  // host-side checks and layouts; a system that fails them gets its status
  // and drops out of the batch
  std::vector<int> live;
  std::vector<Layout> lay(nj);
  std::vector<std::vector<int>> init(nj);
  size_t need = 0;
  int max_it = 1, maxk = 1;
  long idx_total = 0;
  // the differences come after the loop only if no system's threshold can stop it
  bool defer = true;
  for (int j = 0; j < nj; ++j)
    if (spec[j].k >= 1 && spec[j].max_it >= 1)
      defer = defer && can_defer(spec[j].k, spec[j].max_it, spec[j].threshold);
  for (int j = 0; j < nj; ++j) {
    const KmSpec& q = spec[j];
    status[j] = THC_OK;
    if (!q.grid || !q.rho || !q.interp_idx || q.n < 1 || q.k < 1 || q.k > q.n || q.max_it < 1 ||
        q.n > 0x7fffffffL) {
      status[j] = THC_ERR_ARG;
      continue;
    }
    if (q.k > MAXB) {
      status[j] = THC_ERR_UNSUPPORTED;
      continue;
    }
    init[j].resize(q.k);
    if (thc_seed_indices_impl(q.n, q.k, q.seed, init[j].data())) {
      status[j] = THC_ERR_ARG;
      continue;
    }
    lay[j] = plan(q.n, q.k, q.max_it, defer);
    need += bytes_for(lay[j], true);
    max_it = std::max(max_it, q.max_it);
    maxk = std::max(maxk, q.k);
    idx_total += q.k;
    live.push_back(j);
  }
  const int nl = (int)live.size();
  if (nl == 0) return THC_OK;
  // device blob: the job table, the block-count prefix tables, the starting
  // indices; the results block comes back through collect_m
  const size_t job_bytes = align_up(sizeof(Job) * nl, 256);
  const size_t off_bytes = align_up(sizeof(int) * (size_t)JK_COUNT * (nl + 1), 256);
  const size_t idx_bytes = align_up(sizeof(int) * (size_t)idx_total, 256);
  const size_t blob = job_bytes + off_bytes + idx_bytes;
  const long res_stride = (long)align_up(STATE_SLOT + 2 * sizeof(double) * max_it, 64);
  const size_t res_bytes = (size_t)res_stride * nl;
  need += blob + align_up(res_bytes, 256) + 1024;
  if (need > ctx->kmws.cap) {
    if (ctx->kmgraph) ctx->kmgraph->reset();
    THC_TRY(ctx->kmws.reserve(need));
  }
  ctx->kmws.reset();
  char* dblob = ctx->kmws.take<char>(blob);
  char* dres = ctx->kmws.take<char>(res_bytes);
  if (!dblob || !dres) return THC_ERR_NO_MEMORY;
  THC_TRY(ensure_pinned(ctx, std::max(blob, res_bytes)));
  char* hb = reinterpret_cast<char*>(ctx->pinned);
  Job* hj = reinterpret_cast<Job*>(hb);
  int* hoff = reinterpret_cast<int*>(hb + job_bytes);
  int* hidx = reinterpret_cast<int*>(hb + job_bytes + off_bytes);
  int* didx = reinterpret_cast<int*>(dblob + job_bytes + off_bytes);
  long ipos = 0;
  for (int t = 0; t < nl; ++t) {
    const int j = live[t];
    Job& J = hj[t];
    J.L = lay[j];
    if (!carve(ctx->kmws, J.L, J.b, true)) return THC_ERR_NO_MEMORY;
    J.b.idx0 = didx + ipos;  // read by init_run only
    std::copy(init[j].begin(), init[j].end(), hidx + ipos);
    ipos += spec[j].k;
    J.grid = spec[j].grid;
    J.rho = spec[j].rho;
    J.threshold = spec[j].threshold;
    J.interp_idx = spec[j].interp_idx;
  }
  for (int kind = 0; kind < JK_COUNT; ++kind) {
    int* o = hoff + kind * (nl + 1);
    o[0] = 0;
    for (int t = 0; t < nl; ++t) o[t + 1] = o[t] + job_blocks(hj[t].L, kind);
  }
  long total_blocks[JK_COUNT];
  for (int kind = 0; kind < JK_COUNT; ++kind) total_blocks[kind] = hoff[kind * (nl + 1) + nl];
  for (int kind = 0; kind < JK_COUNT; ++kind)
    if (total_blocks[kind] > 0x7fffffffL) return THC_ERR_ARG;
  hipStream_t s = ctx->stream;
  const Job* dj = reinterpret_cast<const Job*>(dblob);
  const int* doff = reinterpret_cast<const int*>(dblob + job_bytes);
  auto off = [&](int kind) { return doff + kind * (nl + 1); };
  auto grid_of = [&](int kind) { return dim3((unsigned)total_blocks[kind]); };
  THC_HIP(hipEventRecord(ctx->ev[0], s));
  THC_HIP(hipMemcpyAsync(dblob, hb, blob, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(init_run_m, grid_of(JK_K256), dim3(256), 0, s, dj, off(JK_K256), nl);
  hipLaunchKernelGGL(bbox_partial_m, grid_of(JK_NBB), dim3(256), 0, s, dj, off(JK_NBB), nl);
  hipLaunchKernelGGL(morton_keys_m, grid_of(JK_N256), dim3(256), 0, s, dj, off(JK_N256), nl);
  hipLaunchKernelGGL(cs_hist_m, grid_of(JK_NCS), dim3(256), 0, s, dj, off(JK_NCS), nl);
  hipLaunchKernelGGL(cs_colscan_m, grid_of(JK_COLSP), dim3(64 * CS_SCAN_W), 0, s, dj, off(JK_COLSP), nl);
  hipLaunchKernelGGL(cs_totscan_m, dim3(nl), dim3(1024), 0, s, dj);
  hipLaunchKernelGGL(cs_scatter_m, grid_of(JK_NCS), dim3(256), 0, s, dj, off(JK_NCS), nl);
  hipLaunchKernelGGL(sorted_tiles_m, grid_of(JK_TILES), dim3(256), 0, s, dj, off(JK_TILES), nl);
  const size_t dyn = (size_t)3 * maxk * sizeof(double);
  for (int it = 0; it < max_it; ++it) {
    with_cpt(maxk, [&](auto cpt) {
      hipLaunchKernelGGL(assign_m<cpt.value>, grid_of(JK_TILES), dim3(256), 0, s, dj, off(JK_TILES), nl, it);
    });
    hipLaunchKernelGGL(centroid_sums_m, grid_of(JK_K), dim3(256), 0, s, dj, off(JK_K), nl, it);
    if (!defer) hipLaunchKernelGGL(diff_control_m, dim3(nl), dim3(1024), dyn, s, dj, it);
  }
  if (defer) {  // beside map_to_grid, as in a single run
    THC_HIP(hipEventRecord(ctx->kev[0], s));
    THC_HIP(hipStreamWaitEvent(ctx->aux, ctx->kev[0], 0));
    for (int it = 0; it < max_it; it += 32768)
      hipLaunchKernelGGL(diff_control_m, dim3(nl, std::min(32768, max_it - it)), dim3(1024), dyn, ctx->aux, dj, it);
    THC_HIP(hipEventRecord(ctx->kev[1], ctx->aux));
  }
  hipLaunchKernelGGL(map_to_grid_m, grid_of(JK_K), dim3(256), 0, s, dj, off(JK_K), nl);
  if (defer) THC_HIP(hipStreamWaitEvent(s, ctx->kev[1], 0));
  hipLaunchKernelGGL(sort_indices_m, dim3(nl), dim3(1024), 0, s, dj);
  hipLaunchKernelGGL(collect_m, dim3(nl), dim3(256), 0, s, dj, dres, res_stride, max_it);
  THC_HIP(hipGetLastError());
  // the pinned buffer still holds the blob being copied: read results back
  // only after that copy (stream order) into the same buffer
  THC_HIP(hipMemcpyAsync(hb, dres, res_bytes, hipMemcpyDeviceToHost, s));
  THC_HIP(hipEventRecord(ctx->ev[1], s));
  THC_HIP(hipStreamSynchronize(s));
  float ms = 0;
  THC_HIP(hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]));
  for (int t = 0; t < nl; ++t) {
    const int j = live[t];
    const char* r = hb + t * res_stride;
    const State* hst = reinterpret_cast<const State*>(r);
    const double* hd = reinterpret_cast<const double*>(r + STATE_SLOT);
    const double* hp = hd + max_it;
    if (stats) {
      thc_kmeans_stats& o = stats[j];
      o.iterations = hst->iters;
      o.converged = hst->mode == MODE_FINAL;
      o.duplicates = hst->dups;
      o.interp_zeroed = hst->mode == MODE_ZEROS;
      o.last_diff = hst->last_diff;
      if (o.diffs) std::copy(hd, hd + hst->iters, o.diffs);
      if (o.pcts) std::copy(hp, hp + hst->iters, o.pcts);
      o.elapsed_ms = ms;
    }
    status[j] = hst->error ? THC_ERR_EMPTY_CLUSTER : (hst->dups ? THC_WARN_DUPLICATE_INDICES : THC_OK);
  }
  return THC_OK;
}

int kmeans_classify(thc_ctx* ctx, const double* grid, long n, const double* centroids, int k, int* grid_map) {
  using namespace km;
  if (!ctx || !grid || !centroids || !grid_map || n < 1 || k < 1 || n > 0x7fffffffL) return THC_ERR_ARG;
  if (k > MAXB) return THC_ERR_UNSUPPORTED;
  THC_HIP(hipSetDevice(ctx->device));
  const Layout L = plan(n, k, 1, false);
  THC_TRY(ctx->ws.reserve(bytes_for(L, false)));
  ctx->ws.reset();
  Bufs b;
  if (!carve(ctx->ws, L, b, false)) return THC_ERR_NO_MEMORY;
  hipStream_t s = ctx->stream;
  enqueue_setup(L, b, grid, s);
  with_cpt(k, [&](auto cpt) {
    hipLaunchKernelGGL(assign<cpt.value>, dim3(L.ntiles), dim3(256), 0, s, b.sx, b.sy, b.sz, b.perm, L.n, b.boxes,
                       b.wboxes, centroids, k, grid_map, (const int*)nullptr, (int*)nullptr, (int*)nullptr, 0,
                       (int2*)nullptr, (int*)nullptr, (int*)nullptr, (const State*)nullptr, 0, -1);
  });
  THC_HIP(hipGetLastError());
  THC_HIP(hipStreamSynchronize(s));
  return THC_OK;
}

int kmeans_update(thc_ctx* ctx, const double* rho, const double* grid, long n, const int* grid_map, int k,
                  double* centroids) {
  using namespace km;
  if (!ctx || !rho || !grid || !grid_map || !centroids || n < 1 || k < 1 || n > 0x7fffffffL) return THC_ERR_ARG;
  if (k > MAXB) return THC_ERR_UNSUPPORTED;
  THC_HIP(hipSetDevice(ctx->device));
  const int cap = bucket_cap(n, k);
  THC_TRY(ctx->ws.reserve(carve_bytes<State>(1) + carve_bytes<int>(k) + carve_bytes<int>((size_t)k * cap) +
                          carve_bytes<int>(4) + carve_bytes<int>(n) + carve_bytes<int2>(n)));
  ctx->ws.reset();
  State* st = ctx->ws.take<State>(1);
  int* cnt = ctx->ws.take<int>(k);
  int* bucket = ctx->ws.take<int>((size_t)k * cap);
  int* ctr = ctx->ws.take<int>(4);
  int* seg = ctx->ws.take<int>(n);
  int2* over = ctx->ws.take<int2>(n);
  if (!st || !cnt || !bucket || !ctr || !seg || !over) return THC_ERR_NO_MEMORY;
  hipStream_t s = ctx->stream;
  hipLaunchKernelGGL(init_run, dim3(ceil_div(k, 256)), dim3(256), 0, s, grid, (const int*)nullptr, k, (double*)nullptr,
                     cnt, ctr, (int*)nullptr, 0, st);
  hipLaunchKernelGGL(bucket_map, dim3(ceil_div(n, CS_TILE)), dim3(256), 0, s, grid_map, n, k, cnt, bucket, cap, over,
                     ctr, st);
  hipLaunchKernelGGL(centroid_sums, dim3(k), dim3(256), 0, s, cnt, bucket, cap, over, ctr, seg, n, rho, grid, centroids,
                     st, 0, -1);
  THC_HIP(hipGetLastError());
  State hst;
  THC_HIP(hipMemcpyAsync(&hst, st, sizeof(State), hipMemcpyDeviceToHost, s));
  THC_HIP(hipStreamSynchronize(s));
  if (hst.error & 2) {
    set_last_error("a grid_map entry lies outside [0, k)", __FILE__, __LINE__);
    return THC_ERR_ARG;
  }
  if (hst.bad == 0) return THC_ERR_EMPTY_CLUSTER;
  return THC_OK;
}

int kmeans_map_to_grid(thc_ctx* ctx, const double* grid, long n, const double* centroids, int k, int* interp_idx) {
  using namespace km;
  if (!ctx || !grid || !centroids || !interp_idx || n < 1 || k < 1 || n > 0x7fffffffL) return THC_ERR_ARG;
  if (k > MAXB) return THC_ERR_UNSUPPORTED;
  THC_HIP(hipSetDevice(ctx->device));
  const Layout L = plan(n, k, 1, false);
  THC_TRY(ctx->ws.reserve(bytes_for(L, false)));
  ctx->ws.reset();
  Bufs b;
  if (!carve(ctx->ws, L, b, false)) return THC_ERR_NO_MEMORY;
  hipStream_t s = ctx->stream;
  hipLaunchKernelGGL(init_run, dim3(1), dim3(256), 0, s, grid, (const int*)nullptr, 0, (double*)nullptr,
                     (int*)nullptr, (int*)nullptr, (int*)nullptr, 0, b.st);
  enqueue_setup(L, b, grid, s);
  hipLaunchKernelGGL(map_to_grid, dim3(k), dim3(256), 0, s, b.sx, b.sy, b.sz, b.perm, L.n, b.boxes, L.ntiles,
                     centroids, 0L, 0, (const State*)nullptr, false, interp_idx);
  hipLaunchKernelGGL(sort_indices, dim3(1), dim3(1024), 0, s, interp_idx, k, b.st);
  THC_HIP(hipGetLastError());
  State hst;
  THC_HIP(hipMemcpyAsync(&hst, b.st, sizeof(State), hipMemcpyDeviceToHost, s));
  THC_HIP(hipStreamSynchronize(s));
  return hst.dups ? THC_WARN_DUPLICATE_INDICES : THC_OK;
}

namespace km {
// y = sqrt(x) with the square root the distance kernels above use
__global__ __launch_bounds__(256) void device_sqrt(const double* x, long n, double* y) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += 256L * gridDim.x) y[i] = sqrt(x[i]);
}
}  // namespace km

}  // namespace thc

extern "C" int thc_device_sqrt(thc_ctx* ctx, const double* x, long n, double* y) {
  using namespace thc;
  if (!ctx || n < 0 || (n > 0 && (!x || !y))) return THC_ERR_ARG;
  if (n == 0) return THC_OK;
  THC_HIP(hipSetDevice(ctx->device));
  const long blocks = std::min<long>(8192, (n + 255) / 256);
  hipLaunchKernelGGL(km::device_sqrt, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, x, n, y);
  THC_HIP(hipGetLastError());
  THC_HIP(hipStreamSynchronize(ctx->stream));
  return THC_OK;
}
