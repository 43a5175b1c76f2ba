// filters.hip -- the steps before ICP: K11 VoxelGrid centroids, K12 statistical
// outlier removal statistics, K13 depth-map back-projection.
//
// K11 replaces pcl::VoxelGrid<PointXYZRGBNormal>::filter with
// setLeafSize(l, l, l) (pcl_tools/cloud_downsampling.cpp:73-75): voxel
// coordinates floor(p * (1/l)) relative to the minimum's, one centroid per
// occupied voxel in increasing voxel index (x fastest).  A stable radix sort of
// (voxel, input index) puts every voxel's points in a run, in input order, and the
// runs in voxel order: a prefix sum over the runs' first points numbers the
// outputs.  Everything is linear in the points, whatever the lattice (a table per
// voxel, with its prefix sums, took 180 us of a 60k-point call at 2 mm) and
// whatever the voxel sizes (with the CLI's default 1 m leaf a whole capture falls
// into a few voxels).  Each run is summed in order (FP32, as PCL's CentroidPoint).
//
// K12 finishes pcl::StatisticalOutlierRemoval (pcl_tools/outlier_removal.cpp:80-84):
// given each point's mean distance to its k nearest neighbours (normals.hip), the
// mean and sample standard deviation over the finite points (FP64, fixed-order
// two-level reduction) and the keep flags.
//
// K13 replaces the depth tool's cross-product normals and back-projection
// (capture/depth_capture/depth_capture.cpp:230-305) for a 16-bit depth map: the
// valid pixels of each 1024-pixel tile are counted, then a block per tile adds the
// counts before its own up, ranks its pixels (row-major output positions) and
// writes points, normals and colours.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <hipcub/hipcub.hpp>

#include "lcr_kernels.hpp"

namespace lcr {

#pragma clang fp contract(off)

namespace {

inline unsigned blocks_of(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

__device__ __forceinline__ bool finite3(const float4& p) {
  return isfinite(p.x) && isfinite(p.y) && isfinite(p.z);
}

// Per point its voxel (skey: nvox for a non-finite point, so that those sort
// last) and its input index (the sort's payload).
__global__ void k_vox_key(const float4* __restrict__ raw, int64_t n, VoxLattice L, int64_t nvox,
                          uint32_t* __restrict__ skey, int* __restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  idx[i] = (int)i;
  const float4 p = raw[i];
  if (!finite3(p)) {
    skey[i] = (uint32_t)nvox;
    return;
  }
  const int ix = (int)(floorf(p.x * L.inv) - (float)L.minb[0]);
  const int iy = (int)(floorf(p.y * L.inv) - (float)L.minb[1]);
  const int iz = (int)(floorf(p.z * L.inv) - (float)L.minb[2]);
  const int64_t k = (int64_t)ix + (int64_t)iy * L.div[0] + (int64_t)iz * L.div[0] * L.div[1];
  skey[i] = (uint32_t)k;
}

// Whether sorted point t is the first of an occupied voxel's run.
__device__ __forceinline__ bool vox_head(const uint32_t* skey, int64_t t, uint32_t nvox) {
  const uint32_t k = skey[t];
  return k < nvox && (t == 0 || skey[t - 1] != k);
}

__global__ void k_vox_heads(const uint32_t* __restrict__ skey, int64_t n, uint32_t nvox,
                            int* __restrict__ heads) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) heads[t] = vox_head(skey, t, nvox) ? 1 : 0;
}

struct VoxCloud {
  const float4 *raw, *nrm;
  const float* curv;
  const uint8_t* rgb;
};
struct VoxOut {
  float *xyz, *nrm, *curv;
  uint8_t* rgb;
};
constexpr int kVoxVals = 10;  // x y z, nx ny nz, curvature, r g b

__device__ __forceinline__ void vox_load(const VoxCloud& in, int64_t i, float (&v)[kVoxVals]) {
  const float4 p = in.raw[i];
  v[0] = p.x;
  v[1] = p.y;
  v[2] = p.z;
  const float4 m = in.nrm ? in.nrm[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  v[3] = m.x;
  v[4] = m.y;
  v[5] = m.z;
  v[6] = in.curv ? in.curv[i] : 0.f;
#pragma unroll
  for (int c = 0; c < 3; ++c) v[7 + c] = in.rgb ? (float)in.rgb[3 * i + c] : 0.f;
}

__device__ __forceinline__ void vox_store(const VoxOut& out, int64_t o, const float (&s)[kVoxVals],
                                          int count) {
  const float cnt = (float)count;
#pragma unroll
  for (int c = 0; c < 3; ++c) out.xyz[3 * o + c] = s[c] / cnt;
  if (out.nrm) {
    // Eigen normalized() of the summed normal: v / sqrt(v . v)
    float nn = s[3] * s[3];
    nn = nn + s[4] * s[4];
    nn = nn + s[5] * s[5];
    const float len = sqrtf(nn);
#pragma unroll
    for (int c = 0; c < 3; ++c) out.nrm[3 * o + c] = len > 0.f ? s[3 + c] / len : s[3 + c];
  }
  if (out.curv) out.curv[o] = s[6] / cnt;
  if (out.rgb) {
#pragma unroll
    for (int c = 0; c < 3; ++c) out.rgb[3 * o + c] = (uint8_t)(uint32_t)(s[7 + c] / cnt);
  }
}

// The centroids, a wavefront per 64 sorted points.  A run that ends within the
// wavefront and holds at most kVoxLaneRun points is summed by its first point's
// lane; a longer one by the whole wavefront: 64 points at a time are loaded
// together into LDS, and a lane per value adds them in order (the same sequence of
// additions).  A lane alone waits for two dependent loads per point, so a run of
// 16 costs it what the wavefront needs for a few hundred points.
constexpr int kVoxLaneRun = 16;
constexpr int kVoxThreads = 256;

__global__ void __launch_bounds__(kVoxThreads)
k_vox_centroid(const uint32_t* __restrict__ skey, const int* __restrict__ idx,
               const int* __restrict__ outidx, int64_t n, uint32_t nvox, VoxCloud in, VoxOut out) {
  __shared__ float stage[kVoxThreads / 64][64][kVoxVals + 1];
  const int lane = threadIdx.x & 63;
  float(*st)[kVoxVals + 1] = stage[threadIdx.x >> 6];
  const int64_t base = ((int64_t)blockIdx.x * kVoxThreads + threadIdx.x) - lane;
  if (base >= n) return;  // uniform across the wavefront
  const int64_t t = base + lane;
  const bool head = t < n && vox_head(skey, t, nvox);
  // where a run may end: at the next head, at the non-finite points, at the end
  const uint64_t stops = __ballot(t >= n || skey[t] >= nvox || head);
  const uint64_t later = lane < 63 ? stops & (~0ull << (lane + 1)) : 0ull;
  const int len = later ? __ffsll((unsigned long long)later) - 1 - lane : kVoxLaneRun + 1;
  if (head && len <= kVoxLaneRun) {
    float s[kVoxVals];
#pragma unroll
    for (int c = 0; c < kVoxVals; ++c) s[c] = 0.f;
    for (int u = 0; u < len; ++u) {
      float v[kVoxVals];
      vox_load(in, idx[t + u], v);
#pragma unroll
      for (int c = 0; c < kVoxVals; ++c) s[c] = s[c] + v[c];
    }
    vox_store(out, outidx[t], s, len);
  }
  for (uint64_t todo = __ballot(head && len > kVoxLaneRun); todo; todo &= todo - 1) {
    const int64_t first = base + __ffsll((unsigned long long)todo) - 1;
    const uint32_t key = skey[first];
    float s = 0.f;
    int64_t count = 0;
    for (int m = 64; m == 64; count += m) {
      const int64_t j = first + count + lane;
      const bool mine = j < n && skey[j] == key;
      m = __popcll(__ballot(mine));
      if (mine) {
        float v[kVoxVals];
        vox_load(in, idx[j], v);
#pragma unroll
        for (int c = 0; c < kVoxVals; ++c) st[lane][c] = v[c];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (lane < kVoxVals) {
#pragma unroll 8
        for (int u = 0; u < m; ++u) s = s + st[u][lane];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    float sums[kVoxVals];
#pragma unroll
    for (int c = 0; c < kVoxVals; ++c) sums[c] = __shfl(s, c, 64);
    if (lane == 0) vox_store(out, outidx[first], sums, (int)count);
  }
}

// K12: block partials of (sum, sum of float squares, finite count) in FP64
constexpr int kSorThreads = 256;

__global__ void __launch_bounds__(kSorThreads)
k_sor_partials(const float* __restrict__ dist, const uint8_t* __restrict__ finite, int64_t n,
               double* __restrict__ part) {
  __shared__ double s0[kSorThreads], s1[kSorThreads], s2[kSorThreads];
  double a = 0.0, b = 0.0, c = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * kSorThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kSorThreads) {
    const float d = dist[i];
    a += d;
    b += (double)(d * d);
    c += finite[i] ? 1.0 : 0.0;
  }
  s0[threadIdx.x] = a;
  s1[threadIdx.x] = b;
  s2[threadIdx.x] = c;
  __syncthreads();
  for (int o = kSorThreads / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s0[threadIdx.x] += s0[threadIdx.x + o];
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[3 * blockIdx.x] = s0[0];
    part[3 * blockIdx.x + 1] = s1[0];
    part[3 * blockIdx.x + 2] = s2[0];
  }
}

// One block: fold the partials in a fixed order; stats = mean, stddev, threshold.
// (One thread adding 391 partials took 50 us of a 100k-point call; this 4.5.)
__global__ void __launch_bounds__(kSorThreads)
k_sor_stats(const double* __restrict__ part, int nparts, double mul, double* __restrict__ stats) {
  __shared__ double s[3][kSorThreads];
  const int t = threadIdx.x;
  double v[3] = {0.0, 0.0, 0.0};
  for (int k = t; k < nparts; k += kSorThreads)
    for (int a = 0; a < 3; ++a) v[a] += part[3 * k + a];
  for (int a = 0; a < 3; ++a) s[a][t] = v[a];
  __syncthreads();
  for (int o = kSorThreads / 2; o > 0; o >>= 1) {
    if (t < o)
      for (int a = 0; a < 3; ++a) s[a][t] += s[a][t + o];
    __syncthreads();
  }
  if (t != 0) return;
  const double sum = s[0][0], sq = s[1][0], valid = s[2][0];
  const double mean = valid > 0.0 ? sum / valid : 0.0;
  const double var = valid > 1.0 ? (sq - sum * sum / valid) / (valid - 1.0) : 0.0;
  const double sd = sqrt(var);
  stats[0] = mean;
  stats[1] = sd;
  stats[2] = mean + mul * sd;
}

__global__ void k_sor_keep(const float* __restrict__ dist, int64_t n, const double* __restrict__ stats,
                           uint8_t* __restrict__ keep) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) keep[i] = (double)dist[i] > stats[2] ? 0 : 1;
}

// K13
__device__ __forceinline__ bool depth_valid(const DepthParams& P, int z, int i, int j) {
  return z != 0 && z >= P.depth_min && z <= P.depth_max && i >= P.top && i <= P.bottom &&
         j >= P.left && j <= P.right;
}

// Valid pixels per tile of kDepthTile pixels: four pixels per thread.  vec: the map
// starts on 8 bytes, so four depths come in one load.
constexpr int kDepthTile = 1024;

__global__ void __launch_bounds__(kDepthTile / 4)
k_depth_count(const uint16_t* __restrict__ depth, int w, int h, DepthParams P, int vec,
              int* __restrict__ counts) {
  __shared__ int s[kDepthTile / 256];
  const int64_t np = (int64_t)w * h;
  const int64_t p = (int64_t)blockIdx.x * kDepthTile + 4 * threadIdx.x;
  int z[4] = {0, 0, 0, 0};
  if (vec && p + 4 <= np) {
    const ushort4 v = *reinterpret_cast<const ushort4*>(depth + p);
    z[0] = v.x;
    z[1] = v.y;
    z[2] = v.z;
    z[3] = v.w;
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (p + u < np) z[u] = depth[p + u];
  }
  int i = (int)(p / w), j = (int)(p % w), c = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    c += __popcll(__ballot(depth_valid(P, z[u], i, j)));  // z = 0 past the end: not valid
    if (++j == w) {
      j = 0;
      ++i;
    }
  }
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

// One pixel per thread, a block per tile.  scanned: counts holds the tiles'
// exclusive scan (then its last entry and the last tile's own count give *out_n);
// else each block adds the counts before its own.
__global__ void __launch_bounds__(kDepthTile)
k_depth_points(const uint16_t* __restrict__ depth, int w, int h, const uint8_t* __restrict__ color,
               DepthParams P, const int* __restrict__ counts, int scanned,
               float* __restrict__ out_xyz, float* __restrict__ out_nrm,
               uint8_t* __restrict__ out_rgb, int64_t* __restrict__ out_n) {
  constexpr int kW = kDepthTile / 64;
  __shared__ int s_before[kW], s_valid[kW];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int64_t np = (int64_t)w * h;
  const int64_t p = (int64_t)blockIdx.x * kDepthTile + t;
  const int i = (int)(p / w), j = (int)(p % w);
  const int z = p < np ? depth[p] : 0;
  const bool valid = depth_valid(P, z, i, j);
  const uint64_t m = __ballot(valid);
  int a = 0;
  if (!scanned)
    for (int k = t; k < (int)blockIdx.x; k += kDepthTile) a += counts[k];
  else if (t == 0)
    a = counts[blockIdx.x];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
  if (lane == 0) {
    s_before[wv] = a;
    s_valid[wv] = __popcll(m);
  }
  __syncthreads();
  int o = 0, total = 0;
#pragma unroll
  for (int k = 0; k < kW; ++k) {
    total += s_before[k] + s_valid[k];
    o += s_before[k] + (k < wv ? s_valid[k] : 0);
  }
  if (t == 0 && blockIdx.x == gridDim.x - 1) *out_n = total;
  if (!valid) return;
  o += __popcll(m & ((1ull << lane) - 1ull));
  int rt = 0, lf = 0, dn = 0, up = 0;
  if (i > 0 && j > 0 && i < h - 1 && j < w - 1) {
    rt = depth[p + w];
    lf = depth[p - w];
    dn = depth[p + 1];
    up = depth[p - 1];
  }
  if (abs(z - rt) > 20) rt = 0;
  if (abs(z - lf) > 20) lf = 0;
  if (abs(z - dn) > 20) dn = 0;
  if (abs(z - up) > 20) up = 0;
  const double dzdx = (rt - lf) / 2.0, dzdy = (dn - up) / 2.0;
  const double vx = -dzdx, vy = -dzdy, vz = 1.0;
  const double inv = 1.0 / sqrt(vx * vx + vy * vy + vz * vz);
  const double px = (double)z * (j - P.cx) * (1 / P.fx);
  const double py = -(double)z * (i - P.cy) * (1 / P.fy);
  const int64_t q = 3 * (int64_t)o;
  out_xyz[q] = (float)px;
  out_xyz[q + 1] = (float)py;
  out_xyz[q + 2] = (float)(-z);
  if (out_nrm) {
    out_nrm[q] = (float)(vx * inv);
    out_nrm[q + 1] = (float)(vy * inv);
    out_nrm[q + 2] = (float)(vz * inv);
  }
  if (out_rgb && color) {
    out_rgb[q] = color[3 * p];
    out_rgb[q + 1] = color[3 * p + 1];
    out_rgb[q + 2] = color[3 * p + 2];
  }
}

}  // namespace

// Bits of the voxel keys the sort looks at: up to nvox (the non-finite marker).
static int vox_key_bits(int64_t nvox) {
  int b = 1;
  while (((int64_t)1 << b) <= nvox) ++b;
  return b;
}

size_t voxel_sort_tmp_bytes(int64_t n, int64_t nvox) {
  size_t bytes = 0;
  if (n <= 0) return 0;
  if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint32_t*)nullptr, (uint32_t*)nullptr,
                                         (const int*)nullptr, (int*)nullptr, (int)n, 0,
                                         vox_key_bits(nvox)) != hipSuccess)
    return 0;
  return bytes;
}

hipError_t launch_voxel_grid(const float4* raw, const float4* raw_nrm, const float* curv,
                             const uint8_t* rgb, int64_t n, const VoxLattice& L, int64_t nvox,
                             VoxScratch w, float* out_xyz, float* out_nrm, float* out_curv,
                             uint8_t* out_rgb, hipStream_t s) {
  if (n <= 0 || nvox <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_vox_key, dim3(blocks_of(n, 256)), dim3(256), 0, s, raw, n, L, nvox, w.skey,
                     w.idx);
  // stable: within a voxel the points keep increasing input index
  size_t bytes = w.sort_tmp_bytes;
  const hipError_t e = hipcub::DeviceRadixSort::SortPairs(w.sort_tmp, bytes, w.skey, w.skey_sorted,
                                                          w.idx, w.sorted_raw, (int)n, 0,
                                                          vox_key_bits(nvox), s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_vox_heads, dim3(blocks_of(n, 256)), dim3(256), 0, s, w.skey_sorted, n,
                     (uint32_t)nvox, w.heads);
  launch_exclusive_scan(w.heads, w.outidx, n, w.scan_tmp, s);
  const VoxCloud in{raw, out_nrm ? raw_nrm : nullptr, out_curv ? curv : nullptr, out_rgb ? rgb : nullptr};
  const VoxOut out{out_xyz, raw_nrm ? out_nrm : nullptr, curv ? out_curv : nullptr, rgb ? out_rgb : nullptr};
  hipLaunchKernelGGL(k_vox_centroid, dim3(blocks_of(n, kVoxThreads)), dim3(kVoxThreads), 0, s,
                     w.skey_sorted, w.sorted_raw, w.outidx, n, (uint32_t)nvox, in, out);
  return hipSuccess;
}

int sor_stat_blocks(int64_t n) {
  const int64_t b = (n + kSorThreads - 1) / kSorThreads;
  return (int)(b < 1 ? 1 : (b > 1024 ? 1024 : b));
}

void launch_sor_stats(const float* dist, const uint8_t* finite, int64_t n, double mul, double* part,
                      double* stats, uint8_t* keep, hipStream_t s) {
  const int nb = sor_stat_blocks(n);
  hipLaunchKernelGGL(k_sor_partials, dim3(nb), dim3(kSorThreads), 0, s, dist, finite, n, part);
  hipLaunchKernelGGL(k_sor_stats, dim3(1), dim3(kSorThreads), 0, s, part, nb, mul, stats);
  if (n > 0)
    hipLaunchKernelGGL(k_sor_keep, dim3(blocks_of(n, 256)), dim3(256), 0, s, dist, n, stats, keep);
}

// Up to this many tiles (4 M pixels) a block adds the counts before its own itself:
// at most four per thread; past it they are scanned first.
constexpr int64_t kDepthInlineTiles = 4096;

int64_t depth_tiles(int64_t pixels) { return (pixels + kDepthTile - 1) / kDepthTile; }

int64_t depth_scratch_ints(int64_t pixels) {
  const int64_t t = depth_tiles(pixels);
  return t <= kDepthInlineTiles ? t : ((t + 3) & ~(int64_t)3) * 2 + scan_tmp_ints(t);
}

void launch_depth_cloud(const uint16_t* depth, int w, int h, const uint8_t* color,
                        const DepthParams& P, int* scratch, float* out_xyz, float* out_nrm,
                        uint8_t* out_rgb, int64_t* out_n, hipStream_t s) {
  const int64_t np = (int64_t)w * h;
  if (np <= 0) return;
  const int64_t tiles = depth_tiles(np), pad = (tiles + 3) & ~(int64_t)3;
  const int vec = (reinterpret_cast<uintptr_t>(depth) & 7) == 0 ? 1 : 0;
  hipLaunchKernelGGL(k_depth_count, dim3((unsigned)tiles), dim3(kDepthTile / 4), 0, s, depth, w, h, P,
                     vec, scratch);
  const bool scanned = tiles > kDepthInlineTiles;
  int* counts = scratch;
  if (scanned) {
    counts = scratch + pad;
    launch_exclusive_scan(scratch, counts, tiles, scratch + 2 * pad, s);
  }
  hipLaunchKernelGGL(k_depth_points, dim3((unsigned)tiles), dim3(kDepthTile), 0, s, depth, w, h, color,
                     P, counts, scanned ? 1 : 0, out_xyz, out_nrm, out_rgb, out_n);
}

}  // namespace lcr
