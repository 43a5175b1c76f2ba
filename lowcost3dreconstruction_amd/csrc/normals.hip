// normals.hip -- K7: k-nearest-neighbour PCA normals.
//
// Replaces pcl::NormalEstimation<PointXYZRGB, Normal>::compute with setKSearch(K)
// (normal_estimation.cpp:84-108): per point, the K nearest neighbours including the
// point itself, their covariance, the eigenvector of the smallest eigenvalue as the
// normal, curvature |l0| / (l0 + l1 + l2), the normal flipped towards the viewpoint
// when (vp - p) . n < 0, then negated when the CLI's flip rule asks
// (normal_estimation.cpp:112-118).  Fewer than 3 neighbours -> NaN normal.
//
// Three selection passes find each point's exact K nearest neighbours by (FLANN
// d2, original index): one lane per query over the 3x3x3 cells around it, one
// wavefront per query that pass leaves over a growing block, and a rescan pass
// with a bisection for what remains.  They sum what the caller needs (FP64 moments
// for the normals, FP64 distances for outlier removal); the solve pass turns the
// moments into normals, one point per lane.
#include <hip/hip_runtime.h>

#include "lcr_common.hpp"
#include "lcr_kernels.hpp"
#include "lcr_math.hpp"
#include "lcr_search.hpp"

namespace lcr {

#pragma clang fp contract(off)

namespace {

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ int popc_ballot(bool p) { return __popcll(__ballot(p)); }

// Number of set bits of b in the lanes below this one.
__device__ __forceinline__ int lane_prefix(uint64_t b) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32),
                                        __builtin_amdgcn_mbcnt_lo((unsigned)b, 0u));
}

struct Moments {
  double v[9];  // sum dx, dy, dz, dx2, dxdy, dxdz, dy2, dydz, dz2 (d = p - q)
};

__device__ __forceinline__ void add_moment(Moments& m, const float4& q, const float4& p) {
  const double dx = (double)p.x - (double)q.x;
  const double dy = (double)p.y - (double)q.y;
  const double dz = (double)p.z - (double)q.z;
  m.v[0] += dx;
  m.v[1] += dy;
  m.v[2] += dz;
  m.v[3] += dx * dx;
  m.v[4] += dx * dy;
  m.v[5] += dx * dz;
  m.v[6] += dy * dy;
  m.v[7] += dy * dz;
  m.v[8] += dz * dz;
}

// What a selection accumulates: kMoments -- FP64 moments of the neighbours
// relative to the query (normals); kSqrtDist -- the sum of sqrt(d2) over the
// neighbours in FP64 (StatisticalOutlierRemoval's mean distance).
constexpr int kMoments = 0;
constexpr int kSqrtDist = 1;

template <int MODE>
__device__ __forceinline__ void take(Moments& m, const float4& q, const float4& p, float d2) {
  if constexpr (MODE == kMoments)
    add_moment(m, q, p);
  else
    m.v[0] += sqrt((double)d2);
}

// A query's sums: nine arrays of n, or one (kSqrtDist).
template <int MODE>
__device__ __forceinline__ void store_sums(const Moments& m, int64_t n, int64_t j, double* mom) {
#pragma unroll
  for (int c = 0; c < (MODE == kMoments ? 9 : 1); ++c) mom[c * n + j] = m.v[c];
}

// One selected point per lane where sel: kMoments writes its original index to
// nbr[base + rank among the wave's selected lanes] (the moments are summed from
// this list by the solve pass); kSqrtDist adds sqrt(d2).  Every lane of the
// wavefront calls it; returns how many lanes selected.
template <int MODE>
__device__ __forceinline__ int select_out(bool sel, const float4& p, unsigned d, const float4& q,
                                          Moments& acc, int* nbr, int base) {
  if constexpr (MODE == kMoments) {
    const uint64_t b = __ballot(sel);
    if (sel) nbr[base + lane_prefix(b)] = __float_as_int(p.w);
    return __popcll(b);
  } else {
    if (sel) take<MODE>(acc, q, p, __uint_as_float(d));
    return 0;
  }
}

// Calls f(j) for this lane's share of the points of rings 0..K.
template <class F>
__device__ __forceinline__ void for_block_points(const GridDesc& g, const int* cs, const CellPos& cp,
                                                 int K, F&& f) {
  const int lane = threadIdx.x & 63;
  for (int ring = 0; ring <= K; ++ring) {
    for_ring_runs(g, cp, ring, [&](int c0, int c1) {
      const int s = cs[c0], e = cs[c1 + 1];
      for (int j = s + lane; j < e; j += 64) f(j);
    });
  }
}

__device__ __forceinline__ int block_count(const GridDesc& g, const int* cs, const CellPos& cp, int K) {
  int total = 0;
  for (int ring = 0; ring <= K; ++ring)
    for_ring_runs(g, cp, ring, [&](int c0, int c1) { total += cs[c1 + 1] - cs[c0]; });
  return total;
}

// Exact path without an LDS buffer: every count rescans the block from memory.
template <int MODE>
__device__ void select_rescan(const GridDesc& g, const int* cs, const float4* pts, const float4& q,
                              const CellPos& cp, int K, int kk, Moments& acc, int* nbr) {
  unsigned T = 0;
  for (;; ++K) {
    const float Lc = block_gap(g, cp, K);
    const bool covers = (Lc == INFINITY);
    if (block_count(g, cs, cp, K) < kk && !covers) continue;
    unsigned lo = 0u, hi = 0x7f800000u;
    while (lo < hi) {
      const unsigned mid = lo + ((hi - lo) >> 1);
      int c = 0;
      for_block_points(g, cs, cp, K, [&](int j) {
        c += (__float_as_uint(flann_d2(q.x, q.y, q.z, pts[j])) <= mid) ? 1 : 0;
      });
      if (wave_sum_i(c) >= kk)
        hi = mid;
      else
        lo = mid + 1;
    }
    T = lo;
    const float L = (Lc - cp.slack) * g.h;
    if (covers || (L > 0.0f && __uint_as_float(T) < L * L * 0.99998f)) break;
  }
  // equal distances at the threshold: keep the smallest original indices
  int clt = 0, cle = 0;
  for_block_points(g, cs, cp, K, [&](int j) {
    const unsigned d = __float_as_uint(flann_d2(q.x, q.y, q.z, pts[j]));
    clt += d < T ? 1 : 0;
    cle += d <= T ? 1 : 0;
  });
  clt = wave_sum_i(clt);
  cle = wave_sum_i(cle);
  int idcut = 0x7fffffff;
  if (cle > kk) {
    const int need = kk - clt;
    unsigned lo = 0u, hi = 0x7fffffffu;
    while (lo < hi) {
      const unsigned mid = lo + ((hi - lo) >> 1);
      int c = 0;
      for_block_points(g, cs, cp, K, [&](int j) {
        const float4 p = pts[j];
        c += (__float_as_uint(flann_d2(q.x, q.y, q.z, p)) == T &&
              (unsigned)__float_as_int(p.w) <= mid)
                 ? 1
                 : 0;
      });
      if (wave_sum_i(c) >= need)
        hi = mid;
      else
        lo = mid + 1;
    }
    idcut = (int)lo;
  }
  // the selected points, in block order (wave-uniform loop: ballot positions)
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int ring = 0; ring <= K; ++ring) {
    for_ring_runs(g, cp, ring, [&](int c0, int c1) {
      const int s = cs[c0], e = cs[c1 + 1];
      for (int jb = s; jb < e; jb += 64) {
        const int j = jb + lane;
        bool sel = false;
        float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
        unsigned d = 0u;
        if (j < e) {
          p = pts[j];
          d = __float_as_uint(flann_d2(q.x, q.y, q.z, p));
          sel = d < T || (d == T && __float_as_int(p.w) <= idcut);
        }
        base += select_out<MODE>(sel, p, d, q, acc, nbr, base);
      }
    });
  }
}

// ---------------------------------------------------------------- lane path
//
// One query per lane (64 neighbouring cell-sorted queries per wavefront, each
// lane on its own): the candidates are the points of the (2K+1)^3 cells around
// the query's cell, read from memory (the wavefront's queries share most of
// them, so the reads hit the caches).  The kk-th smallest FLANN d2 is certified
// when it lies below D2, the squared distance from the query to the block's
// boundary (minus the rounding slack), so only d2 < D2 counts, and each row of
// the block is trimmed to the cells that can hold such a point (ball_row).  Pass 1 builds a
// per-lane histogram of d2 over [0, D2) in NB equal buckets -- on a surface the
// number of points within a radius grows with its square, so the buckets fill
// about evenly -- and finds the bucket B that holds the kk-th.  Pass 2 lists
// the positions of the points of lower buckets and of bucket B's in LDS; a sorting
// network orders bucket B's by (d2, original index) and the first kk - (count
// below B) complete the list.  Bucket index =
// floor(d2 * scale) is monotone in d2, so the result is exactly the kk smallest
// (d2, original index).  A query is flagged for the next path when its block
// covers the grid, holds fewer than kk points under D2 (not certified), more
// than kLaneMaxCand candidates, or more than NL points in bucket B.
//
// The lane pass runs K = 1 (3x3x3 cells) over every point and appends the
// points it flags (a few percent: near crop edges and silhouettes the 3x3x3
// block holds too few; dense spots overflow bucket B) to a list, which the
// wavefront pass below serves.
constexpr int kLaneMaxCand = 4096;
// The lane pass's histogram buckets (the wavefront pass reads its bucket bounds
// in units of D2 / kLaneBuckets).
constexpr int kLaneBuckets = 32;

constexpr int kLaneThreads = 256;

// Sorted-array start and length of the (2K+1)^2 x-runs (at most 2K+1 cells each)
// of the block of radius K around cp: the cell-table loads are issued together.
template <int K>
struct BlockRuns {
  static constexpr int R = (2 * K + 1) * (2 * K + 1);
  int s[R], n[R];
};

// The cells of row (z, y) of the block of radius K that may hold a point with d2
// below D2: [xa, xb] (empty when xa > xb).  Each cell's lower-bound distance per
// axis is axis_gap (cell units, less the rounding slack), and the bound is
// widened by 2e-5 for the float rounding of d2, as the ring search prunes.
__device__ __forceinline__ void ball_row(const GridDesc& g, const CellPos& cp, int K, int z, int y,
                                         float D2, int& xa, int& xb) {
  const float gz = axis_gap(cp.fz, z, cp.cz, cp.slack), gy = axis_gap(cp.fy, y, cp.cy, cp.slack);
  const float thr = D2 * 1.00002f;
  const float lyz = (gz * gz + gy * gy) * (g.h * g.h);
  const float dxc = sqrtf(fmaxf(thr - lyz, 0.0f)) * g.inv_h * 1.00001f + cp.slack;
  xa = max(max(cp.cx - K, (int)ceilf(cp.fx - dxc - 1.0f)), 0);
  xb = min(min(cp.cx + K, (int)floorf(cp.fx + dxc)), g.nx - 1);
  if (z < 0 || z >= g.nz || y < 0 || y >= g.ny || lyz > thr) xb = xa - 1;
}

// The runs of the block of radius K trimmed to the cells that may hold a point
// with d2 below D2 (ball_row): only those can count towards the certificate.
template <int K>
__device__ __forceinline__ BlockRuns<K> block_runs(const GridDesc& g, const int* cs, const CellPos& cp,
                                                   float D2) {
  BlockRuns<K> b;
#pragma unroll
  for (int r = 0; r < BlockRuns<K>::R; ++r) {
    const int z = cp.cz + r / (2 * K + 1) - K, y = cp.cy + r % (2 * K + 1) - K;
    int xa, xb;
    ball_row(g, cp, K, z, y, D2, xa, xb);
    const bool in = xa <= xb;
    const int row = in ? (z * g.ny + y) * g.nx : 0;
    const int s = in ? cs[row + xa] : 0;
    const int e = in ? cs[row + xb + 1] : 0;
    b.s[r] = s;
    b.n[r] = e - s;
  }
  return b;
}

// The cell-sorted points as a raw buffer (gfx9 resource word 3): a load is one
// 32-bit offset add, and a load past the end returns zeros instead of faulting.
// The caller keeps n * 16 below 2^31 bytes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t points_rsrc(const float4* pts, int64_t n) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)pts, (short)0, (int)(n * 16), 0x00020000);
}

__device__ __forceinline__ float4 load_point(__amdgpu_buffer_rsrc_t r, int i) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, i * 16, 0, 0));
}

// Calls f(p, i, valid) for the points i of the block's runs, NBATCH loads in
// flight; the loads of a run's last batch read on past its end (the next points,
// or zeros past the buffer) with valid = false.  The runs go column by column:
// the 2K+1 runs of one y offset (z = -K .. K) back to back, each lane moving to
// its next non-empty run as soon as it finishes one.  A loop over one run at a
// time lasts as long as the wavefront's longest lane in every run; per column,
// the lanes' long and short runs even out (about 76 against 101 batches per
// wavefront on the 36-capture cycle's queries).  after() follows every batch.
template <int K, int NBATCH, class F, class G>
__device__ __forceinline__ void for_block(const BlockRuns<K>& b, __amdgpu_buffer_rsrc_t rs, F&& f,
                                          G&& after) {
  constexpr int S = 2 * K + 1;
#pragma unroll
  for (int dy = 0; dy < S; ++dy) {
    // the column's runs with the empty ones moved to the end, order kept
    int qs[S], qe[S];
#pragma unroll
    for (int t = 0; t < S; ++t) {
      qs[t] = b.s[t * S + dy];
      qe[t] = qs[t] + b.n[t * S + dy];
    }
#pragma unroll
    for (int pass = 0; pass + 1 < S; ++pass)
#pragma unroll
      for (int t = 0; t + 1 < S; ++t) {
        const bool gap = qs[t] >= qe[t];
        qs[t] = gap ? qs[t + 1] : qs[t];
        qe[t] = gap ? qe[t + 1] : qe[t];
        qs[t + 1] = gap ? 0 : qs[t + 1];
        qe[t + 1] = gap ? 0 : qe[t + 1];
      }
    int i = qs[0], e = qe[0];
    while (i < e) {
      float4 p[NBATCH];
#pragma unroll
      for (int u = 0; u < NBATCH; ++u) p[u] = load_point(rs, i + u);
#pragma unroll
      for (int u = 0; u < NBATCH; ++u) f(p[u], i + u, i + u < e);
      after();
      i += NBATCH;
      if (i >= e) {
        i = qs[1];
        e = qe[1];
#pragma unroll
        for (int t = 1; t + 1 < S; ++t) {
          qs[t] = qs[t + 1];
          qe[t] = qe[t + 1];
        }
        qs[S - 1] = 0;
        qe[S - 1] = 0;
      }
    }
  }
}

// (key, payload) compare-exchange: smaller key first.
__device__ __forceinline__ void cswap(uint64_t& a, uint64_t& b, int& pa, int& pb) {
  const bool sw = b < a;
  const uint64_t lo = sw ? b : a, hi = sw ? a : b;
  const int plo = sw ? pb : pa, phi = sw ? pa : pb;
  a = lo;
  b = hi;
  pa = plo;
  pb = phi;
}

// Sorts NL (key, payload) pairs: the 19-comparator network for 8, odd-even
// transposition (NL rounds) otherwise.
template <int NL>
__device__ __forceinline__ void sort_keys(uint64_t (&e)[NL], int (&ei)[NL]) {
  if constexpr (NL == 8) {
    cswap(e[0], e[2], ei[0], ei[2]); cswap(e[1], e[3], ei[1], ei[3]);
    cswap(e[4], e[6], ei[4], ei[6]); cswap(e[5], e[7], ei[5], ei[7]);
    cswap(e[0], e[4], ei[0], ei[4]); cswap(e[1], e[5], ei[1], ei[5]);
    cswap(e[2], e[6], ei[2], ei[6]); cswap(e[3], e[7], ei[3], ei[7]);
    cswap(e[0], e[1], ei[0], ei[1]); cswap(e[2], e[3], ei[2], ei[3]);
    cswap(e[4], e[5], ei[4], ei[5]); cswap(e[6], e[7], ei[6], ei[7]);
    cswap(e[2], e[4], ei[2], ei[4]); cswap(e[3], e[5], ei[3], ei[5]);
    cswap(e[1], e[4], ei[1], ei[4]); cswap(e[3], e[6], ei[3], ei[6]);
    cswap(e[1], e[2], ei[1], ei[2]); cswap(e[3], e[4], ei[3], ei[4]); cswap(e[5], e[6], ei[5], ei[6]);
  } else {
#pragma unroll
    for (int round = 0; round < NL; ++round)
#pragma unroll
      for (int t = round & 1; t + 1 < NL; t += 2) cswap(e[t], e[t + 1], ei[t], ei[t + 1]);
  }
}

// Block b of n runs on XCD b % 8 (the hardware's round-robin); this returns the
// logical block such that each XCD takes one contiguous range of them, so that
// neighbouring cell-sorted queries -- and the cells they read -- share an L2.
__device__ __forceinline__ int xcd_block(int b, int n) {
  const int x = b & 7, slot = b >> 3, q = n >> 3, rem = n & 7;
  return x * q + min(x, rem) + slot;
}

template <int NB, int NL>
constexpr int lane_words() {
  return 2 * NL > NB ? 2 * NL : NB;
}

// nsel bit: the query's list holds original indices into the cloud's raw points
// (the rescan path), not positions in the cell-sorted copy.
constexpr int kNselOrig = 1 << 30;

// One query of the lane path. K: block radius in cells; NB: histogram buckets;
// NL: bucket-B capacity; buf: the lane's LDS column (lane_words words).  Writes
// the FP64 moments of the selected neighbours relative to the query (mom, nine
// arrays of n) and nsel, and returns 0; or leaves the query to the next path
// (nothing written) and returns the block radius that path starts from: K + 1
// when this block held too few points or no certificate, K otherwise; when
// bucket B overflowed, B + 1 in bits 8 and up (at least kk points lie below
// (B + 1) D2 / NB, up to the rounding of d2 * scale).
template <int MODE, int K, int NB, int NL>
__device__ __forceinline__ int lane_query(const GridDesc* __restrict__ grids,
                                          const int* __restrict__ cell_start,
                                          const float4* __restrict__ pts,
                                          __amdgpu_buffer_rsrc_t rs,
                                          const int* __restrict__ cloud_of_sorted, int k, int64_t j,
                                          uint32_t (*buf)[64], int lane, double* __restrict__ mom,
                                          int64_t n, int* __restrict__ nsel) {
  const float4 q = pts[j];
  const GridDesc g = grids[cloud_of_sorted[j]];
  const int kk = min(k, g.npts);
  if (MODE == kMoments && kk < 3) {
    nsel[j] = kk;
    return 0;
  }
  const int* cs = cell_start + g.cell_off;
  const CellPos cp = cell_pos(g, q.x, q.y, q.z);
  const float Lc = block_gap(g, cp, K);
  const float L = (Lc - cp.slack) * g.h;
  const float D2 = L * L * 0.99998f;
  const float scale = (float)NB / D2;
  // blocks that cover the grid (no boundary to certify against) and gaps inside
  // the rounding slack go on; a finite scale keeps every bucket index of a
  // d2 < D2 inside [0, NB]
  if (!(Lc < INFINITY && L > 0.0f && D2 > 1e-30f && scale < INFINITY)) return K;
  const BlockRuns<K> blk = block_runs<K>(g, cs, cp, D2);
  int m = 0;
#pragma unroll
  for (int r = 0; r < BlockRuns<K>::R; ++r) m += blk.n[r];
  if (m < kk) return K + 1;
  if (m > kLaneMaxCand) return K;
#pragma unroll
  for (int c = 0; c < NB; ++c) buf[c][lane] = 0u;
  // pass 1, branch-free: every candidate adds 0 or 1 to its bucket
  for_block<K, 4>(blk, rs, [&](const float4& p, int, bool valid) {
    const float d = flann_d2(q.x, q.y, q.z, p);
    const int b = (int)fminf(d * scale, (float)(NB - 1));
    atomicAdd(&buf[b][lane], (valid && d < D2) ? 1u : 0u);
  }, [] {});
  int B = -1, below = 0, nB = 0, cum = 0;
  // four counts at a time: unrolled whole, the 32 reads would all be in flight
#pragma unroll 4
  for (int c = 0; c < NB; ++c) {
    const int v = (int)buf[c][lane];
    if (B < 0 && cum + v >= kk) {
      B = c;
      below = cum;
      nB = v;
    }
    cum += v;
  }
  if (B < 0) return K + 1;  // not certified
  if (nB > NL) return K | ((B + 1) << 8);
  // Pass 2 takes points of buckets up to B only: floor(d2 * scale) <= B < NB - 1
  // means d2 < (B + 1) D2 / NB, to within the rounding of d2 * scale (1e-4 covers
  // it).  The rows trimmed to that bound (ball_row, monotone in the bound) keep
  // every such point, and their runs are sub-runs of pass 1's, so the points
  // pass 2 takes and the order it adds them in are unchanged.
  const BlockRuns<K> sel =
      B < NB - 1 ? block_runs<K>(g, cs, cp, fminf(D2, D2 * ((float)(B + 1) / (float)NB) * 1.0001f))
                 : blk;
  // the moments of the lower buckets' points in block order, then of bucket B's
  // picks in (d2, original index) order.  The block's scan only writes positions to
  // the lane's column: lower buckets' to rows 0 .. kList - 1, bucket B's to the last
  // NL (at most nB of them).  The moments are then added over the list, where nearly
  // every lane has a point in every step; added in the scan, each of its steps ran
  // the FP64 sums for the few lanes whose point was in (62 % of the pass).  A slot
  // that is not taken leaves its position at the row the next one overwrites.
  // bucket < B: d2 * scale < B; bucket B: below B + 1, or the last one.
  constexpr int kList = lane_words<NB, NL>() - NL;
  static_assert(kList >= 8, "a list of two batches at least");
  const float fB = (float)B, fB1 = B < NB - 1 ? (float)(B + 1) : INFINITY;
  Moments acc;
#pragma unroll
  for (int c = 0; c < 9; ++c) acc.v[c] = 0.0;
  int na = 0, nl = 0;
  auto flush = [&] {
    for (int t = 0; t < na; t += 4) {
      float4 p[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) p[u] = load_point(rs, t + u < na ? (int)buf[t + u][lane] : 0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (t + u < na) take<MODE>(acc, q, p[u], flann_d2(q.x, q.y, q.z, p[u]));
    }
    na = 0;
  };
  for_block<K, 4>(
      sel, rs,
      [&](const float4& p, int i, bool valid) {
        const float d = flann_d2(q.x, q.y, q.z, p);
        const float x = d * scale;
        const bool lower = x < fB;
        const bool in = valid & (d < D2) & (x < fB1);
        const int row = in & !lower ? kList + nl : na;
        buf[row][lane] = (uint32_t)i;
        na += in & lower ? 1 : 0;
        nl += in & !lower ? 1 : 0;
      },
      [&] {
        if (__any(na > kList - 4)) flush();
      });
  flush();
  uint64_t e[NL];
  int ei[NL];
#pragma unroll
  for (int t = 0; t < NL; ++t) {
    ei[t] = t < nl ? (int)buf[kList + t][lane] : 0;
    const float4 p = load_point(rs, ei[t]);
    const uint64_t key =
        ((uint64_t)__float_as_uint(flann_d2(q.x, q.y, q.z, p)) << 32) | (uint32_t)__float_as_int(p.w);
    e[t] = t < nl ? key : ~0ull;
  }
  sort_keys<NL>(e, ei);
  const int need = kk - below;
#pragma unroll
  for (int t = 0; t < NL; ++t)
    if (t < need) {
      if constexpr (MODE == kMoments)
        add_moment(acc, q, load_point(rs, ei[t]));
      else
        take<MODE>(acc, q, q, __uint_as_float((uint32_t)(e[t] >> 32)));
    }
  store_sums<MODE>(acc, n, j, mom);
  if constexpr (MODE == kMoments) nsel[j] = kk;
  return 0;
}

// Appends the lanes where take holds to list (list[*count ...]: the point and
// the block radius to start from), one atomic per wavefront; every lane of the
// wavefront calls it.  The order of the list depends on scheduling; every
// consumer's result per query does not.
__device__ __forceinline__ void wave_append(bool take, int64_t j, int start_k,
                                            int2* __restrict__ list, int* __restrict__ count) {
  const uint64_t b = __ballot(take);
  if (b == 0) return;
  const int lead = __ffsll((unsigned long long)b) - 1;
  int base = 0;
  if ((int)(threadIdx.x & 63) == lead) base = atomicAdd(count, __popcll(b));
  base = __builtin_amdgcn_readlane(base, lead);
  if (take) list[base + lane_prefix(b)] = make_int2((int)j, start_k);
}

// The lane pass over every point: one lane per point, blocks mapped
// XCD-contiguous; the points it leaves are appended to list.  No barrier: each
// lane uses only its own LDS column.
template <int MODE, int K, int NB, int NL>
__global__ void __launch_bounds__(kLaneThreads)
k_normal_lane(const GridDesc* __restrict__ grids, const int* __restrict__ cell_start,
              const float4* __restrict__ pts, const int* __restrict__ cloud_of_sorted,
              int64_t total, int k, double* __restrict__ mom, int* __restrict__ nsel,
              int2* __restrict__ list, int* __restrict__ count) {
  static_assert(NB == kLaneBuckets, "the wavefront pass reads bucket bounds of kLaneBuckets");
  __shared__ uint32_t s_buf[kLaneThreads / 64][lane_words<NB, NL>()][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t j = (int64_t)xcd_block(blockIdx.x, gridDim.x) * kLaneThreads + threadIdx.x;
  const __amdgpu_buffer_rsrc_t rs = points_rsrc(pts, total);
  const int start_k = j < total ? lane_query<MODE, K, NB, NL>(grids, cell_start, pts, rs, cloud_of_sorted,
                                                        k, j, s_buf[w], lane, mom, total, nsel)
                                : 0;
  wave_append(start_k > 0, j, start_k, list, count);
}

// ---------------------------------------------------------------- wavefront pass
//
// The queries the lane pass leaves, one wavefront per query.  The candidates are
// the (2K+1)^2 x-runs of the block of radius K around the query's cell, each
// trimmed to the cells that can hold a point below D2 (ball_row), taken 64 runs
// at a time; the lanes stride through each chunk's points together (consecutive
// lanes read consecutive points of a run).
//
// Pass 1 counts d2 < D2 (the block's certified range, as in the lane path) in
// kWaveBuckets equal buckets of a histogram the wavefront shares in LDS.  Fewer
// than kk below D2 means the kk-th neighbour may lie outside the block; any kk
// of the block's points bound its distance from above (the kk-th smallest of the
// per-lane minima, distinct points, or the largest d2 when fewer lanes hold one),
// and the next block is the smallest whose certified range holds that bound, so
// it certifies.  That bound (or, for a query whose lane-pass bucket overflowed,
// the bound of that bucket) then narrows the histogram's range: at least kk
// points lie below it, so counting d2 < R2 = min(D2, bound) over the rows
// trimmed to R2 finds the same kk nearest with fewer candidates and finer
// buckets.  A prefix over the buckets gives bucket B of the kk-th; more
// than 64 points in B split it into 256 sub-buckets with one more pass (the
// bucket key floor(256 * d2 * scale) at that level, still monotone in d2).
// Pass 2 adds the points of lower keys to the lane's FP64 moments (each lane its
// share of the block, in block order) and keeps the kk-th's key's entries (d2,
// original index, position) in LDS, where each one's rank among them picks the
// first kk - (count below); a wavefront sum in a fixed order then gives the
// query's moments.  The selected set is exactly the kk smallest (d2, original
// index).  A block that covers the grid holds every point and certifies itself;
// a radius above kWaveMaxK or more than 64 equal keys sends the query to the
// rescan pass.
constexpr int kWaveBuckets = 256;
constexpr int kWaveMaxK = 48;
constexpr int kWaveThreads = 256;

struct WaveLds {
  int hist[kWaveBuckets];
  int pref[65];  // points before run r of the chunk
  int start[64]; // run r's first sorted position
  uint32_t key[64], idx[64];
  int pos[64];
};

// Inclusive prefix sum over the wavefront.
__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// The kk-th smallest of the lanes' values (ties by lane), kk <= 64.
__device__ __forceinline__ float wave_kth_smallest(float v, int kk) {
  const int lane = threadIdx.x & 63;
  int rank = 0;
  for (int u = 0; u < 64; ++u) {
    const float w = __shfl(v, u, 64);
    rank += (w < v || (w == v && u < lane)) ? 1 : 0;
  }
  const int at = __ffsll((unsigned long long)__ballot(rank == kk - 1)) - 1;
  return __shfl(v, at, 64);
}

// Calls f(valid, p, i) for this lane's share of the points of the block of radius
// K that may lie below D2 (i: the sorted position; rows trimmed by ball_row), run
// chunk by run chunk; every lane takes part in every call (valid = false past a
// chunk's end), so f may use ballots.
template <class F>
__device__ __forceinline__ void for_wave_block(WaveLds& L, const GridDesc& g, const int* cs,
                                               const CellPos& cp, int K, float D2,
                                               __amdgpu_buffer_rsrc_t rs, F&& f) {
  const int lane = threadIdx.x & 63;
  const int side = 2 * K + 1, R = side * side;
  for (int r0 = 0; r0 < R; r0 += 64) {
    const int r = r0 + lane;
    int st = 0, len = 0;
    if (r < R) {
      const int z = cp.cz + r / side - K, y = cp.cy + r % side - K;
      int xa, xb;
      ball_row(g, cp, K, z, y, D2, xa, xb);
      if (xa <= xb) {
        const int row = (z * g.ny + y) * g.nx;
        st = cs[row + xa];
        len = cs[row + xb + 1] - st;
      }
    }
    const int incl = wave_incl_scan(len);
    const int total = __shfl(incl, 63, 64);
    if (total == 0) continue;
    wave_lds_sync();  // the previous chunk's reads are done
    L.start[lane] = st;
    L.pref[lane + 1] = incl;
    if (lane == 0) L.pref[0] = 0;
    wave_lds_sync();
    // two points per lane in flight; t past the chunk's end maps to position 0
    // (loaded, not used)
    int rr = 0;
    for (int base = 0; base < total; base += 128) {
      const int t0 = base + lane, t1 = t0 + 64;
      const bool v0 = t0 < total, v1 = t1 < total;
      int i0 = 0, i1 = 0;
      if (v0) {
        while (t0 >= L.pref[rr + 1]) ++rr;  // runs may be empty
        i0 = L.start[rr] + (t0 - L.pref[rr]);
      }
      if (v1) {
        while (t1 >= L.pref[rr + 1]) ++rr;
        i1 = L.start[rr] + (t1 - L.pref[rr]);
      }
      const float4 p0 = load_point(rs, i0), p1 = load_point(rs, i1);
      f(v0, p0, i0);
      f(v1, p1, i1);
    }
  }
}

// Bucket B of the kk-th among the counts in L.hist (lane l holds buckets 4l ..
// 4l + 3) plus `below` points before them: returns false when the counts hold
// fewer than kk; otherwise B, the count before B (below updated) and B's count.
__device__ __forceinline__ bool wave_find_bucket(const WaveLds& L, int kk, int& below, int& B,
                                                 int& nB) {
  const int lane = threadIdx.x & 63;
  int h[4], sum = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    h[c] = L.hist[4 * lane + c];
    sum += h[c];
  }
  const int incl = wave_incl_scan(sum) + below;
  if (__shfl(incl, 63, 64) < kk) return false;
  const bool cross = incl >= kk && incl - sum < kk;
  const int cl = __ffsll((unsigned long long)__ballot(cross)) - 1;
  int b = 0, bl = 0, n = 0;
  if (cross) {
    int cum = incl - sum;
    b = -1;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (b < 0 && cum + h[c] >= kk) {
        b = 4 * lane + c;
        bl = cum;
        n = h[c];
      }
      cum += h[c];
    }
  }
  B = __builtin_amdgcn_readlane(b, cl);
  below = __builtin_amdgcn_readlane(bl, cl);
  nB = __builtin_amdgcn_readlane(n, cl);
  return true;
}

// An upper bound of the distance from a query inside the grid to any of its points.
__device__ __forceinline__ float grid_extent(const GridDesc& g) {
  return ((float)g.nx + (float)g.ny + (float)g.nz + 3.0f) * g.h;
}

template <int MODE>
__global__ void __launch_bounds__(kWaveThreads, 5)
k_normal_wave(const GridDesc* __restrict__ grids, const int* __restrict__ cell_start,
              const float4* __restrict__ pts, const int* __restrict__ cloud_of_sorted, int k,
              const int2* __restrict__ list, const int* __restrict__ count, int64_t total,
              double* __restrict__ mom, int* __restrict__ nsel, int* __restrict__ deferred) {
  __shared__ WaveLds s_w[kWaveThreads / 64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  WaveLds& L = s_w[w];
  const int n = *count;
  const int nwaves = (int)gridDim.x * (kWaveThreads / 64);
  const __amdgpu_buffer_rsrc_t rs = points_rsrc(pts, total);
  for (int qi = (int)blockIdx.x * (kWaveThreads / 64) + w; qi < n; qi += nwaves) {
    const int2 e = list[qi];
    const int64_t j = __builtin_amdgcn_readfirstlane(e.x);
    const float4 q = pts[j];
    const GridDesc g = grids[cloud_of_sorted[j]];
    const int kk = min(k, g.npts);  // kMoments: at least 3, the lane pass serves the others
    const int* cs = cell_start + g.cell_off;
    const CellPos cp = cell_pos(g, q.x, q.y, q.z);
    bool done = false;
    const int code = __builtin_amdgcn_readfirstlane(e.y);
    int K = code & 0xff;
    // a d2 that at least kk points lie below (INFINITY: none known yet)
    float U = INFINITY;
    for (int attempt = 0; attempt < 8 && !done && K <= kWaveMaxK; ++attempt) {
      const float Lc = block_gap(g, cp, K);
      // A block that covers the grid holds every point and needs no certificate: its
      // range is the grid's extent
      const float Lm = Lc == INFINITY ? grid_extent(g) : (Lc - cp.slack) * g.h;
      const float D2 = Lm * Lm * 0.99998f;
      // the lane pass's bucket bound (same block, same D2), widened for rounding
      if (attempt == 0 && (code >> 8) > 0)
        U = D2 * ((float)(code >> 8) / (float)kLaneBuckets) * 1.0001f;
      // The passes count d2 < R2: the certified range, or U below it.  The kk
      // nearest then lie below R2, and the rows trimmed to R2 hold them.
      const float R2 = (U > 1e-30f && U < D2) ? U : D2;
      const float scale = (float)kWaveBuckets / R2;
      if (!(Lm > 0.0f && D2 > 1e-30f && scale < INFINITY)) {
        ++K;
        continue;
      }
      wave_lds_sync();
#pragma unroll
      for (int c = lane; c < kWaveBuckets; c += 64) L.hist[c] = 0;
      // pass 1: the histogram of d2 < R2, and the lane's count, least and largest d2
      int mc = 0;
      float dmin = INFINITY, dmax = 0.0f;
      for_wave_block(L, g, cs, cp, K, R2, rs, [&](bool valid, const float4& p, int) {
        if (!valid) return;
        const float d = flann_d2(q.x, q.y, q.z, p);
        ++mc;
        dmin = fminf(dmin, d);
        dmax = fmaxf(dmax, d);
        if (d < R2) atomicAdd(&L.hist[min((int)(d * scale), kWaveBuckets - 1)], 1);
      });
      wave_lds_sync();
      if (wave_sum_i(mc) < kk) {
        K = 2 * K + 1;
        continue;
      }
      int below = 0, B, nB;
      if (!wave_find_bucket(L, kk, below, B, nB)) {
        // not certified: a block whose certified range holds an upper bound U of
        // the kk-th d2 certifies (its gap is at least its radius in cells)
        const float Ub = (kk <= 64 && popc_ballot(mc > 0) >= kk) ? wave_kth_smallest(dmin, kk)
                                                                  : wave_max_f(dmax);
        const float need = sqrtf(Ub) * g.inv_h * 1.0001f + cp.slack + 1e-3f;
        K = max(K + 1, (int)ceilf(fminf(need, (float)(kWaveMaxK + 1))));
        U = fminf(U, Ub * 1.0001f);  // kk points of this block lie at or below Ub
        continue;
      }
      // The passes below take points of keys up to bucket B only: floor(d2 *
      // scale) <= B < kWaveBuckets - 1 means d2 < (B + 1) R2 / kWaveBuckets, to
      // within the rounding of d2 * scale (1e-4 covers it), so they walk the rows
      // trimmed to that bound (ball_row keeps every cell that may hold such a
      // point).
      const float D2b = B < kWaveBuckets - 1
                            ? fminf(R2, R2 * ((float)(B + 1) / (float)kWaveBuckets) * 1.0001f)
                            : R2;
      // level 1 inside bucket B when it holds more than 64 points
      int SB = 0;
      const bool split = nB > 64;
      if (split) {
        wave_lds_sync();
#pragma unroll
        for (int c = lane; c < kWaveBuckets; c += 64) L.hist[c] = 0;
        wave_lds_sync();
        for_wave_block(L, g, cs, cp, K, D2b, rs, [&](bool valid, const float4& p, int) {
          if (!valid) return;
          const float d = flann_d2(q.x, q.y, q.z, p);
          if (!(d < R2)) return;
          const float x = d * scale;
          if (min((int)x, kWaveBuckets - 1) != B) return;
          atomicAdd(&L.hist[min((int)((x - (float)B) * 256.0f), 255)], 1);
        });
        wave_lds_sync();
        wave_find_bucket(L, kk, below, SB, nB);
        if (nB > 64) break;  // more than 64 equal keys: the rescan pass
      }
      // pass 2: the moments of the lower keys, the kk-th's key kept in LDS; with
      // the split, keys up to (B, SB) lie below (B + (SB + 1) / 256) R2 /
      // kWaveBuckets (x - B and its product by 256 are exact)
      const float D2s =
          split && B < kWaveBuckets - 1
              ? fminf(D2b, R2 * (((float)B + (float)(SB + 1) * (1.0f / 256.0f)) / (float)kWaveBuckets) *
                               1.0001f)
              : D2b;
      Moments acc;
#pragma unroll
      for (int c = 0; c < 9; ++c) acc.v[c] = 0.0;
      int nl = 0;
      for_wave_block(L, g, cs, cp, K, D2s, rs, [&](bool valid, const float4& p, int i) {
        const float d = valid ? flann_d2(q.x, q.y, q.z, p) : INFINITY;
        const float x = d * scale;
        const int b = d < R2 ? min((int)x, kWaveBuckets - 1) : kWaveBuckets;
        const int sb = (split && b == B) ? min((int)((x - (float)B) * 256.0f), 255) : 0;
        const bool lt = b < B || (b == B && sb < SB);
        const bool eq = b == B && sb == SB;
        const uint64_t beq = __ballot(eq);
        if (lt) take<MODE>(acc, q, p, d);
        if (eq) {
          const int slot = nl + lane_prefix(beq);
          L.key[slot] = __float_as_uint(d);
          L.idx[slot] = (uint32_t)__float_as_int(p.w);
          L.pos[slot] = i;
        }
        nl += __popcll(beq);
      });
      wave_lds_sync();
      // rank of each kept entry by (d2, original index): unique keys
      if (lane < nl) {
        const uint64_t mine = ((uint64_t)L.key[lane] << 32) | L.idx[lane];
        int rank = 0;
        for (int u = 0; u < nl; ++u) rank += (((uint64_t)L.key[u] << 32) | L.idx[u]) < mine ? 1 : 0;
        if (rank < kk - below) {
          if constexpr (MODE == kMoments)
            add_moment(acc, q, load_point(rs, L.pos[lane]));
          else
            take<MODE>(acc, q, q, __uint_as_float(L.key[lane]));
        }
      }
#pragma unroll
      for (int c = 0; c < (MODE == kMoments ? 9 : 1); ++c) acc.v[c] = wave_sum_dpp(acc.v[c]);
      if (lane == 0) {
        store_sums<MODE>(acc, total, j, mom);
        if constexpr (MODE == kMoments) nsel[j] = kk;
      }
      done = true;
    }
    if (!done && lane == 0) {
      // deferred[0] counts the list deferred[1..]
      if constexpr (MODE == kMoments) nsel[j] = kk | kNselOrig;
      deferred[1 + atomicAdd(deferred, 1)] = (int)j;
    }
    wave_lds_sync();  // L is reused by the next query
  }
}

// Rescan pass for the deferred queries (see the wavefront pass), one
// wavefront per query, reading the block from memory for every count.
template <int MODE>
__global__ void __launch_bounds__(256)
k_normal_rescan(const GridDesc* __restrict__ grids, const int* __restrict__ cell_start,
                const float4* __restrict__ pts, const int* __restrict__ cloud_of_sorted, int k,
                const int* __restrict__ deferred, double* __restrict__ mom, int* __restrict__ nbr) {
  const int lane = threadIdx.x & 63;
  const int nwaves = (int)(gridDim.x * (blockDim.x >> 6));
  const int count = deferred[0];
  for (int wi = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)); wi < count;
       wi += nwaves) {
    const int64_t j = deferred[1 + wi];
    const float4 q = pts[j];
    const GridDesc g = grids[cloud_of_sorted[j]];
    const int kk = min(k, g.npts);
    Moments acc;
#pragma unroll
    for (int i = 0; i < 9; ++i) acc.v[i] = 0.0;
    select_rescan<MODE>(g, cell_start + g.cell_off, pts, q, cell_pos(g, q.x, q.y, q.z), 1, kk, acc,
                        MODE == kMoments ? nbr + j * k : nullptr);
    if constexpr (MODE == kSqrtDist) {
      const double s = wave_sum_dpp(acc.v[0]);
      if (lane == 0) mom[j] = s;
    }
  }
}

// Solve pass, one point per lane: the FP64 moments of its neighbours relative to
// it (from the lane and wavefront passes, or summed here in list order from the
// rescan pass's list of original indices, kNselOrig set), covariance, normal
// (eigenvector of the smallest eigenvalue, FP64) oriented towards the viewpoint.
// Bound by FP64 latency: 36 captures (37k-113k points each) 211 us with Jacobi for every point,
// 64 with the closed form; four wavefronts a SIMD for it (8 spills) over two.
__global__ void __launch_bounds__(256, 4)
k_normal_solve(const float4* __restrict__ pts, const int* __restrict__ cloud_of_sorted,
               const float4* __restrict__ raw, const int64_t* __restrict__ cloud_off,
               const int* __restrict__ nbr, int k, const double* __restrict__ mom,
               const int* __restrict__ nsel, int64_t total, const float* __restrict__ vp,
               int flip_all, float4* __restrict__ out) {
  const int64_t jq = (int64_t)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (jq >= total) return;
  const int ns = nsel[jq];
  const int cnt = ns & ~kNselOrig;
  if (cnt < 3) {
    out[jq] = make_float4(NAN, NAN, NAN, NAN);
    return;
  }
  const float4 q = pts[jq];
  Moments acc;
  if (ns & kNselOrig) {
    const float4* R = raw + cloud_off[cloud_of_sorted[jq]];
    const int* list = nbr + jq * k;
#pragma unroll
    for (int i = 0; i < 9; ++i) acc.v[i] = 0.0;
    for (int i = 0; i < cnt; ++i) add_moment(acc, q, R[list[i]]);
  } else {
#pragma unroll
    for (int i = 0; i < 9; ++i) acc.v[i] = mom[i * total + jq];
  }
  const double* m = acc.v;
  const double n = (double)cnt;
  const double mx = m[0] / n, my = m[1] / n, mz = m[2] / n;
  double C[3][3];
  C[0][0] = m[3] / n - mx * mx;
  C[0][1] = m[4] / n - mx * my;
  C[0][2] = m[5] / n - mx * mz;
  C[1][1] = m[6] / n - my * my;
  C[1][2] = m[7] / n - my * mz;
  C[2][2] = m[8] / n - mz * mz;
  C[1][0] = C[0][1];
  C[2][0] = C[0][2];
  C[2][1] = C[1][2];
  const float* v = vp + 3 * cloud_of_sorted[jq];
  const double ex = (double)v[0] - q.x, ey = (double)v[1] - q.y, ez = (double)v[2] - q.z;
  const double sum = C[0][0] + C[1][1] + C[2][2];
  double w0, e[3];
  bool ok = smallest_eigvec3(C, w0, e);
  double dot = ex * e[0] + ey * e[1] + ez * e[2];
  // (a normal square to the view keeps the sign that Jacobi gives it)
  if (!ok || !(fabs(dot) > 0.0)) {
    double wv[3], V[3][3];
    eigh3(C, wv, V);
    w0 = wv[0];
#pragma unroll
    for (int i = 0; i < 3; ++i) e[i] = V[i][0];
    dot = ex * e[0] + ey * e[1] + ez * e[2];
  }
  double nx = e[0], ny = e[1], nz = e[2];
  const double curv = sum != 0.0 ? fabs(w0 / sum) : 0.0;
  if (dot < 0.0) {
    nx = -nx;
    ny = -ny;
    nz = -nz;
  }
  if (flip_all) {
    nx = -nx;
    ny = -ny;
    nz = -nz;
  }
  out[jq] = make_float4((float)nx, (float)ny, (float)nz, (float)curv);
}

// StatisticalOutlierRemoval's value per input point: sum / mean_k in FP64 rounded
// to float at the point's input position; finite flag for the statistics.
__global__ void k_sor_dist(const float4* __restrict__ pts, const int* __restrict__ cloud_of_sorted,
                           const int64_t* __restrict__ cloud_off, const double* __restrict__ sums,
                           int64_t total, int mean_k, float* __restrict__ dist,
                           uint8_t* __restrict__ finite) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= total) return;
  const int64_t i = cloud_off[cloud_of_sorted[j]] + __float_as_int(pts[j].w);
  dist[i] = (float)(sums[j] / (double)mean_k);
  finite[i] = 1;
}

}  // namespace

int64_t normals_work_ints(int64_t n) { return 4 * n + 3; }

// The selection passes over every point: sums (and, kMoments, nsel and the rescan
// pass's neighbour lists).  work (normals_work_ints(n)): [0] the lane pass's list
// count, [1] the rescan count with its list at [2, 2 + n), the lane pass's list of
// (point, start radius) at [2 + n, 2 + 3n).
template <int MODE>
static void launch_selection(const GridDesc* grids, const int* cell_start, const float4* pts,
                             const int* cloud_of_sorted, int64_t n, int k, int* nbr, double* mom,
                             int* nsel, int* work, hipStream_t s) {
  int* count = work;
  int* deferred = work + 1;
  int2* list = reinterpret_cast<int2*>(work + 2 + n + (n & 1));
  launch_fill_i32(work, 2, 0, s);
  hipLaunchKernelGGL((k_normal_lane<MODE, 1, kLaneBuckets, 8>),
                     dim3((unsigned)((n + kLaneThreads - 1) / kLaneThreads)), dim3(kLaneThreads), 0, s,
                     grids, cell_start, pts, cloud_of_sorted, n, k, mom, nsel, list, count);
  // persistent over the list (a few percent of the points): at most eight blocks
  // of four wavefronts per CU
  const int64_t wave_blocks = (n + kWaveThreads / 64 - 1) / (kWaveThreads / 64);
  hipLaunchKernelGGL(k_normal_wave<MODE>, dim3((unsigned)(wave_blocks < 2048 ? wave_blocks : 2048)),
                     dim3(kWaveThreads), 0, s, grids, cell_start, pts, cloud_of_sorted, k,
                     (const int2*)list, (const int*)count, n, mom, nsel, deferred);
  hipLaunchKernelGGL(k_normal_rescan<MODE>, dim3(1024), dim3(256), 0, s, grids, cell_start, pts,
                     cloud_of_sorted, k, deferred, mom, nbr);
}

// Outlier removal runs the same selection as the normals, summing distances: 100k
// points, 50 neighbours: 1477 -> 249 us against one wavefront per query over a
// block staged in LDS.
void launch_sor_distances(const GridDesc* grids, const int* cell_start, const float4* pts,
                          const int* cloud_of_sorted, const int64_t* cloud_off, int64_t npts_total,
                          int mean_k, double* sums, int* work, float* dist, uint8_t* finite,
                          hipStream_t s) {
  if (npts_total <= 0) return;
  launch_selection<kSqrtDist>(grids, cell_start, pts, cloud_of_sorted, npts_total, mean_k + 1, nullptr,
                              sums, nullptr, work, s);
  hipLaunchKernelGGL(k_sor_dist, dim3((unsigned)((npts_total + 255) / 256)), dim3(256), 0, s, pts,
                     cloud_of_sorted, cloud_off, sums, npts_total, mean_k, dist, finite);
}

void launch_normals(const GridDesc* grids, const int* cell_start, const float4* pts,
                    const int* cloud_of_sorted, int64_t npts_total, int k, const float* vp,
                    int flip_all, const float4* raw, const int64_t* cloud_off, int* nbr, double* mom,
                    int* nsel, int* work, float4* nrm_sorted, hipStream_t s) {
  if (npts_total <= 0) return;
  const int64_t n = npts_total;
  launch_selection<kMoments>(grids, cell_start, pts, cloud_of_sorted, n, k, nbr, mom, nsel, work, s);
  hipLaunchKernelGGL(k_normal_solve, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, pts,
                     cloud_of_sorted, raw, cloud_off, nbr, k, (const double*)mom, nsel, n, vp,
                     flip_all, nrm_sorted);
}

}  // namespace lcr
