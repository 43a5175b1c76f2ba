// runtime.cpp -- host runtime of liblcr (see runtime.hpp).
#include "runtime.hpp"

#include "lcr_search.hpp"

#include <atomic>
#include <thread>

#include <float.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>

namespace lcr {

// ------------------------------------------------------------------ profiler

Profiler& Profiler::get() {
  static Profiler p;
  return p;
}

hipEvent_t Profiler::take() {
  if (!pool_.empty()) {
    hipEvent_t e = pool_.back();
    pool_.pop_back();
    return e;
  }
  hipEvent_t e;
  LCR_HIP(hipEventCreate(&e));
  return e;
}

void Profiler::reset() {
  std::lock_guard<std::mutex> g(mu_);
  totals_.clear();
}

int Profiler::begin(const char* name, hipStream_t s, std::vector<Span>* into) {
  if (!on_ || !into) return -1;
  std::lock_guard<std::mutex> g(mu_);
  Span sp{name, take(), take()};
  LCR_HIP(hipEventRecord(sp.a, s));
  into->push_back(sp);
  return (int)into->size() - 1;
}

void Profiler::end(int span, hipStream_t s, std::vector<Span>* into) {
  if (span < 0 || !into) return;
  LCR_HIP(hipEventRecord((*into)[span].b, s));
}

void Profiler::collect(std::vector<Span>& spans, bool keep) {
  std::lock_guard<std::mutex> g(mu_);
  for (auto& sp : spans) {
    LCR_HIP(hipEventSynchronize(sp.b));
    float ms = 0.f;
    LCR_HIP(hipEventElapsedTime(&ms, sp.a, sp.b));
    auto& t = totals_[sp.name];
    t.first += 1;
    t.second += ms;
    if (!keep) {
      pool_.push_back(sp.a);
      pool_.push_back(sp.b);
    }
  }
  if (!keep) spans.clear();
}

bool Profiler::read(const std::string& name, int64_t* launches, double* ms) {
  std::lock_guard<std::mutex> g(mu_);
  auto it = totals_.find(name);
  if (it == totals_.end()) {
    *launches = 0;
    *ms = 0.0;
    return false;
  }
  *launches = it->second.first;
  *ms = it->second.second;
  return true;
}

int device_cu_count() {
  int dev = 0;
  LCR_HIP(hipGetDevice(&dev));
  int cus = 0;
  LCR_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return cus > 0 ? cus : 1;
}

// ------------------------------------------------------------------ copies

CopyOut::~CopyOut() {
  for (hipEvent_t e : done_)
    if (e) (void)hipEventDestroy(e);
}

void CopyOut::add(void* dst, const void* src, size_t bytes) {
  for (size_t at = 0; at < bytes;) {
    if (filled_ == kChunk) {
      first_.push_back(pieces_.size());
      filled_ = 0;
    }
    const size_t len = std::min(kChunk - filled_, bytes - at);
    pieces_.push_back(Piece{static_cast<char*>(dst) + at, static_cast<const char*>(src) + at, len, filled_});
    filled_ += len;
    at += len;
  }
}

// A chunk that has arrived goes to the caller.
void CopyOut::move(size_t chunk) {
  const char* in = stage_.as<char>() + chunk % kSlots * kChunk;
  const size_t end = chunk + 1 < first_.size() ? first_[chunk + 1] : pieces_.size();
  for (size_t k = first_[chunk]; k < end; ++k) memcpy(pieces_[k].dst, in + pieces_[k].off, pieces_[k].bytes);
}

void CopyOut::finish() {
  const size_t n = first_.size();
  if (n > 0) stage_.reserve(n == 1 ? filled_ : std::min<size_t>(n, kSlots) * kChunk);
  size_t moved = 0;
  auto arrive = [&] {  // the oldest chunk under way
    LCR_HIP(hipEventSynchronize(done_[moved % kSlots]));
    move(moved++);
  };
  for (size_t c = 0; c < n; ++c) {
    if (c >= (size_t)kSlots) arrive();  // its place in the ring
    char* to = stage_.as<char>() + c % kSlots * kChunk;
    const size_t end = c + 1 < n ? first_[c + 1] : pieces_.size();
    for (size_t k = first_[c]; k < end; ++k)
      LCR_HIP(hipMemcpyAsync(to + pieces_[k].off, pieces_[k].src, pieces_[k].bytes, hipMemcpyDeviceToHost,
                             s_));
    if (c + 1 == n) break;  // the wait for the stream covers the last one
    hipEvent_t& e = done_[c % kSlots];
    if (!e) LCR_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    LCR_HIP(hipEventRecord(e, s_));
  }
  while (moved + 1 < n) arrive();
  LCR_HIP(hipStreamSynchronize(s_));
  if (moved < n) move(moved);
}

void copy_in(hipStream_t s, void* dst, const void* src, size_t bytes, HostBuf& stage) {
  if (bytes == 0) return;
  if (bytes <= kCopyInStage) {
    stage.reserve(bytes);
    memcpy(stage.p, src, bytes);
    src = stage.p;
  }
  LCR_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
}

// ------------------------------------------------------------------ clouds

namespace {

__global__ void k_segments(const int64_t* __restrict__ off, int n, int64_t total,
                           int* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  int lo = 0, hi = n - 1;
  while (lo < hi) {  // last segment whose start is <= i
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= i)
      lo = mid;
    else
      hi = mid - 1;
  }
  out[i] = lo;
}

void launch_segments(const int64_t* off, int n, int64_t total, int* out, hipStream_t s) {
  if (total <= 0) return;
  hipLaunchKernelGGL(k_segments, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, off, n,
                     total, out);
}

constexpr int64_t kMaxDim = 4096;

}  // namespace

// Host threads staging an upload, and the points below which one thread does it.
constexpr int kStageThreads = 8;
constexpr int64_t kStageMinPoints = 1 << 18;

// The records are packed to 12 bytes a point in pinned memory, copied over in one
// go, and widened on the device (with each point's cloud), so 12 bytes a point
// cross the bus instead of 20 and the host only copies.
void CloudSet::upload(hipStream_t s, const std::vector<const float*>& xyz,
                      const std::vector<const float*>& nrm, const std::vector<int64_t>& counts,
                      int64_t stride_bytes, bool zero_nrm, bool pinned) {
  n = (int)xyz.size();
  geom_valid = false;
  nraw = counts;
  raw_off.assign(n + 1, 0);
  for (int c = 0; c < n; ++c) raw_off[c + 1] = raw_off[c] + counts[c];
  total_raw = raw_off[n];
  int with = 0;
  for (int c = 0; c < n; ++c) with += nrm[c] ? 1 : 0;
  has_nrm = zero_nrm ? with > 0 : with == n;
  const size_t np = (size_t)std::max<int64_t>(total_raw, 1);
  const int parts = has_nrm ? 2 : 1;  // points, then normals
  LCR_HIP(hipStreamSynchronize(s));  // the last upload is done with its buffers
  d_in.reserve(np * 3 * sizeof(float) * parts);
  float* din[2] = {d_in.as<float>(), d_in.as<float>() + 3 * np};
  d_raw.reserve(np * sizeof(float4));
  d_point_cloud.reserve(np * sizeof(int));
  if (has_nrm) d_raw_nrm.reserve(np * sizeof(float4));
  d_cloud_off.reserve((n + 1) * sizeof(int64_t));
  h_small.reserve((n + 1) * sizeof(int64_t) + 4096);
  memcpy(h_small.p, raw_off.data(), (n + 1) * sizeof(int64_t));
  LCR_HIP(hipMemcpyAsync(d_cloud_off.p, h_small.p, (n + 1) * sizeof(int64_t),
                         hipMemcpyHostToDevice, s));
  if (pinned) {
    for (int c = 0; c < n; ++c) {
      const size_t len = (size_t)counts[c] * 3 * sizeof(float);
      if (len == 0) continue;
      LCR_HIP(hipMemcpyAsync(din[0] + 3 * raw_off[c], xyz[c], len, hipMemcpyHostToDevice, s));
      if (!has_nrm) continue;
      if (nrm[c])
        LCR_HIP(hipMemcpyAsync(din[1] + 3 * raw_off[c], nrm[c], len, hipMemcpyHostToDevice, s));
      else
        launch_fill_i32(reinterpret_cast<int*>(din[1] + 3 * raw_off[c]), 3 * counts[c], 0, s);
    }
  } else {
    h_stage.reserve(np * 3 * sizeof(float) * parts);
    float* st[2] = {h_stage.as<float>(), h_stage.as<float>() + 3 * np};
    auto stage = [&](int c) {
      for (int q = 0; q < parts; ++q) {
        const char* in = reinterpret_cast<const char*>(q == 0 ? xyz[c] : nrm[c]);
        float* o = st[q] + 3 * raw_off[c];
        if (counts[c] == 0) continue;
        if (!in) {
          memset(o, 0, (size_t)counts[c] * 3 * sizeof(float));
        } else if (stride_bytes == 3 * (int64_t)sizeof(float)) {
          memcpy(o, in, (size_t)counts[c] * 3 * sizeof(float));
        } else {
          for (int64_t i = 0; i < counts[c]; ++i) memcpy(o + 3 * i, in + i * stride_bytes, 3 * sizeof(float));
        }
      }
    };
    const int nthreads = (int)std::min<int64_t>(
        {(int64_t)kStageThreads, (int64_t)n, std::max<int64_t>(total_raw / kStageMinPoints, 1)});
    if (nthreads <= 1) {
      for (int c = 0; c < n; ++c) stage(c);
    } else {
      std::atomic<int> next{0};
      std::vector<std::thread> pool;
      for (int t = 0; t < nthreads; ++t)
        pool.emplace_back([&] {
          for (int c = next++; c < n; c = next++) stage(c);
        });
      for (std::thread& th : pool) th.join();
    }
    for (int q = 0; q < parts; ++q)
      if (total_raw > 0)
        LCR_HIP(hipMemcpyAsync(din[q], st[q], (size_t)total_raw * 3 * sizeof(float),
                               hipMemcpyHostToDevice, s));
  }
  launch_segments(d_cloud_off.as<int64_t>(), n, total_raw, d_point_cloud.as<int>(), s);
  launch_widen(din[0], has_nrm ? din[1] : nullptr, total_raw, d_raw.as<float4>(),
               has_nrm ? d_raw_nrm.as<float4>() : nullptr, s);
}

namespace {
// Disjoint regions of the pinned scratch used by one grid build (async copies of
// different regions may be in flight together).
struct BuildRegions {
  size_t geom, grids, poff, total;
  explicit BuildRegions(int n) {
    auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
    geom = 0;
    grids = al(geom + (size_t)n * kGeomWords * sizeof(float));
    poff = al(grids + (size_t)n * sizeof(GridDesc));
    total = al(poff + (size_t)(n + 1) * sizeof(int64_t));
  }
};
}  // namespace

CloudSet::~CloudSet() {
  if (ev_build) (void)hipEventDestroy(ev_build);
  if (ev_vp) (void)hipEventDestroy(ev_vp);
}

void CloudSet::build(hipStream_t s, double factor, std::vector<Profiler::Span>* spans,
                     bool with_tree, int stage) {
  const bool from_normals = stage == kBuildFromNormals;
  // the sorted input's layout (finite points per cloud) comes from the same upload
  if (from_normals && !geom_valid) throw Error{-5, "no normals-stage build to start from"};
  // the previous build's copies out of the pinned region must be done
  if (ev_build)
    LCR_HIP(hipEventSynchronize(ev_build));
  else
    LCR_HIP(hipEventCreateWithFlags(&ev_build, hipEventDisableTiming));
  Profiler& prof = Profiler::get();
  if (factor <= 0.0) factor = 2.5;
  const BuildRegions R(n);
  h_build.reserve(R.total);
  char* hb = h_build.as<char>();
  GridDesc* hg = reinterpret_cast<GridDesc*>(hb + R.grids);
  int64_t* hpoff = reinterpret_cast<int64_t*>(hb + R.poff);
  const int span = prof.begin("grid_build", s, spans);
  // 1. bounding boxes, finite counts and the probe grids' (<= 65 cells on the longest
  //    axis) occupied cells depend only on the uploaded points: measured once per
  //    upload, in one go
  d_grids.reserve((size_t)n * sizeof(GridDesc));
  if (!geom_valid) {
    d_bbox_part.reserve((size_t)n * kBBoxChunks * 7 * sizeof(float));
    d_geom.reserve((size_t)n * kGeomWords * sizeof(float));
    d_probe.reserve((size_t)n * kProbeWords * sizeof(uint32_t));
    launch_bbox(d_raw.as<float4>(), d_cloud_off.as<int64_t>(), n, d_bbox_part.as<float>(),
                d_geom.as<float>(), d_grids.as<GridDesc>(), d_probe.as<uint32_t>(), s);
    launch_probe(d_raw.as<float4>(), d_cloud_off.as<int64_t>(), d_grids.as<GridDesc>(), n,
                 d_probe.as<uint32_t>(), d_geom.as<float>(), s);
    float* hgeom = reinterpret_cast<float*>(hb + R.geom);
    LCR_HIP(hipMemcpyAsync(hgeom, d_geom.p, (size_t)n * kGeomWords * sizeof(float),
                           hipMemcpyDeviceToHost, s));
    LCR_HIP(hipStreamSynchronize(s));
    geom.assign(hgeom, hgeom + (size_t)n * kGeomWords);
    geom_valid = true;
    d_in.release();  // the upload is done with them
    h_stage.release();
  }

  // 2. the probe grids
  grids.assign(n, GridDesc{});
  for (int c = 0; c < n; ++c) {
    grids[c] = probe_grid(&geom[(size_t)c * kGeomWords]);
    grids[c].nraw = (int)nraw[c];
  }
  d_cid.reserve((size_t)std::max<int64_t>(total_raw, 1) * sizeof(int));
  d_place.reserve((size_t)std::max<int64_t>(total_raw, 1) * sizeof(int));

  // 3. final cell edge: factor * spacing, spacing ~ h0 / sqrt(points per occupied
  //    probe cell) for surface-sampled clouds; capped cell count and extent
  int64_t cells = 0;
  total_pts = 0;
  for (int c = 0; c < n; ++c) {
    GridDesc& g = grids[c];
    const float* b = &geom[(size_t)c * kGeomWords];
    int occ;
    memcpy(&occ, b + 7, sizeof occ);
    g.pt_off = total_pts;
    total_pts += g.npts;
    if (g.npts > 0) {
      const double h0 = g.h;
      const double per_cell = (double)g.npts / std::max(occ, 1);
      const double spacing = h0 / sqrt(std::max(per_cell, 1.0));
      double h = std::max(factor * spacing, 1e-6);
      const double ex = (double)b[3] - b[0], ey = (double)b[4] - b[1], ez = (double)b[5] - b[2];
      const double max_cells = std::max<double>(16.0 * g.npts, 4096.0);
      for (int it = 0; it < 64; ++it) {
        const double nx = floor(ex / h) + 1, ny = floor(ey / h) + 1, nz = floor(ez / h) + 1;
        if (nx <= kMaxDim && ny <= kMaxDim && nz <= kMaxDim && nx * ny * nz <= max_cells) break;
        h *= 1.25;
      }
      g.h = (float)h;
      g.inv_h = (float)(1.0 / (double)g.h);
      g.nx = (int)(floor(ex * (double)g.inv_h) + 1);
      g.ny = (int)(floor(ey * (double)g.inv_h) + 1);
      g.nz = (int)(floor(ez * (double)g.inv_h) + 1);
    }
    g.cell_off = cells;
    g.near_r = 0.0f;
    g.near_off = 0;
    cells += (int64_t)g.nx * g.ny * g.nz + 1;
  }
  if (cells > (int64_t)1 << 30) throw Error{-5, "grid too large"};
  total_cells = cells;
  // bounding-volume trees: leaves of kLeaf sorted points, complete binary tree
  int64_t nodes = 0;
  max_depth = 0;
  for (int c = 0; c < n; ++c) {
    GridDesc& g = grids[c];
    const int64_t leaves = (g.npts + kLeaf - 1) / kLeaf;
    int d = 0;
    while (((int64_t)1 << d) < leaves) ++d;
    g.depth = d;
    g.node_off = nodes;
    nodes += (int64_t)2 << d;  // 1-based heap: indices 1 .. 2^(d+1) - 1
    max_depth = std::max(max_depth, d);
  }
  total_nodes = nodes;
  memcpy(hg, grids.data(), (size_t)n * sizeof(GridDesc));
  LCR_HIP(hipMemcpyAsync(d_grids.p, hg, (size_t)n * sizeof(GridDesc), hipMemcpyHostToDevice, s));

  // 4. count, scan, scatter, per-cell sort.  The counters are zero over the whole
  // allocation between builds (the scan consumes the counts), so they are filled
  // only after a reallocation.
  if (d_counts.reserve((size_t)cells * sizeof(int))) counts_zero = false;
  d_cell_start.reserve((size_t)cells * sizeof(int));
  d_scan_tmp.reserve((size_t)scan_tmp_ints(cells) * sizeof(int));
  const size_t npts = (size_t)std::max<int64_t>(total_pts, 1);
  DevBuf& out_pts = stage == kBuildNormals ? d_npts : d_pts;
  DevBuf& out_nrm = stage == kBuildNormals ? d_nnrm : d_nrm;
  out_pts.reserve(npts * sizeof(float4));
  out_nrm.reserve(npts * sizeof(float4));
  d_cloud_of_sorted.reserve(npts * sizeof(int));
  // input: the upload, or the normals stage's sorted points (finite only, the
  // clouds in the same order) with the normals computed on them
  const float4* in_pts = from_normals ? d_npts.as<float4>() : d_raw.as<float4>();
  const float4* in_nrm = from_normals ? d_nnrm.as<float4>()
                                      : (has_nrm ? d_raw_nrm.as<float4>() : nullptr);
  const int* in_cloud = from_normals ? d_cloud_of_sorted.as<int>() : d_point_cloud.as<int>();
  const int64_t n_in = from_normals ? total_pts : total_raw;
  if (!counts_zero) launch_fill_i32(d_counts.as<int>(), (int64_t)(d_counts.bytes / sizeof(int)), 0, s);
  counts_zero = false;
  launch_cell_count(in_pts, in_cloud, d_grids.as<GridDesc>(), n_in, d_cid.as<int>(),
                    d_counts.as<int>(), d_place.as<int>(), s);
  launch_exclusive_scan_consume(d_counts.as<int>(), d_cell_start.as<int>(), cells,
                                d_scan_tmp.as<int>(), s);
  d_slot_raw.reserve(npts * sizeof(int));
  d_slot_cell.reserve(npts * sizeof(int));
  launch_place_points(in_pts, in_nrm, d_cid.as<int>(), d_place.as<int>(), n_in, total_pts,
                      d_cell_start.as<int>(), d_slot_raw.as<int>(), d_slot_cell.as<int>(),
                      d_cloud_off.as<int64_t>(), d_point_cloud.as<int>(), out_pts.as<float4>(),
                      out_nrm.as<float4>(), from_normals, s);
  if (from_normals) has_nrm = true;
  counts_zero = true;
  // sorted point -> cloud
  for (int c = 0; c < n; ++c) hpoff[c] = grids[c].pt_off;
  hpoff[n] = total_pts;
  d_poff.reserve((size_t)(n + 1) * sizeof(int64_t));
  LCR_HIP(hipMemcpyAsync(d_poff.p, hpoff, (n + 1) * sizeof(int64_t), hipMemcpyHostToDevice, s));
  launch_segments(d_poff.as<int64_t>(), n, total_pts, d_cloud_of_sorted.as<int>(), s);
  // tree order, then the bounding-volume tree over it
  if (!with_tree) {
    prof.end(span, s, spans);
    LCR_HIP(hipEventRecord(ev_build, s));  // the pinned regions are reused by the next build
    return;
  }
  d_tpts.reserve(npts * sizeof(float4));
  d_tpos.reserve(npts * sizeof(int));
  d_tkeys.reserve(npts * sizeof(uint64_t));
  d_tkeys_sorted.reserve(npts * sizeof(uint64_t));
  d_tvals.reserve(npts * sizeof(int));
  if (ttmp_pts != total_pts || ttmp_n != n) {  // the size query is slow: once per shape
    ttmp_bytes = tree_order_tmp_bytes(total_pts, n);
    ttmp_pts = total_pts;
    ttmp_n = n;
  }
  const size_t tmp_bytes = ttmp_bytes;
  d_ttmp.reserve(std::max<size_t>(tmp_bytes, 16));
  LCR_HIP(launch_tree_order(d_grids.as<GridDesc>(), n, d_pts.as<float4>(), d_cloud_of_sorted.as<int>(),
                            total_pts, d_tkeys.as<uint64_t>(), d_tkeys_sorted.as<uint64_t>(),
                            d_tvals.as<int>(), d_tpos.as<int>(), d_ttmp.p, tmp_bytes,
                            d_tpts.as<float4>(), s));
  d_nodes.reserve((size_t)std::max<int64_t>(total_nodes, 1) * 2 * sizeof(float4));
  launch_bvh_build(d_grids.as<GridDesc>(), n, max_depth, d_tpts.as<float4>(), d_nodes.as<float4>(), s);
  prof.end(span, s, spans);
  LCR_HIP(hipEventRecord(ev_build, s));  // the pinned regions are reused by the next build
}

void CloudSet::compute_normals(hipStream_t s, int k, const float* vp_host, int flip_all,
                               std::vector<Profiler::Span>* spans, bool normals_stage) {
  Profiler& prof = Profiler::get();
  // the previous pass's copy out of h_vp must be done before it is rewritten
  if (ev_vp)
    LCR_HIP(hipEventSynchronize(ev_vp));
  else
    LCR_HIP(hipEventCreateWithFlags(&ev_vp, hipEventDisableTiming));
  d_vp.reserve((size_t)n * 3 * sizeof(float));
  h_vp.reserve((size_t)n * 3 * sizeof(float));
  float* v = h_vp.as<float>();
  for (int c = 0; c < n; ++c)
    for (int a = 0; a < 3; ++a) v[3 * c + a] = vp_host ? vp_host[3 * c + a] : 0.0f;
  LCR_HIP(hipMemcpyAsync(d_vp.p, v, (size_t)n * 3 * sizeof(float), hipMemcpyHostToDevice, s));
  LCR_HIP(hipEventRecord(ev_vp, s));
  // the selection reads the sorted points through a raw buffer of 32-bit byte offsets
  if (total_pts > ((int64_t)1 << 27) - 1) throw Error{-5, "more than 2^27 points in one normals batch"};
  const int span = prof.begin("normals", s, spans);
  const size_t np = (size_t)std::max<int64_t>(total_pts, 1);
  d_nbr.reserve(np * (size_t)k * sizeof(int));
  d_nsel.reserve(np * sizeof(int));
  d_nmom.reserve(np * 9 * sizeof(double));
  d_nwork.reserve((size_t)normals_work_ints((int64_t)np) * sizeof(int));
  DevBuf& pts = normals_stage ? d_npts : d_pts;
  DevBuf& nrm = normals_stage ? d_nnrm : d_nrm;
  nrm.reserve(np * sizeof(float4));
  launch_normals(d_grids.as<GridDesc>(), d_cell_start.as<int>(), pts.as<float4>(),
                 d_cloud_of_sorted.as<int>(), total_pts, k, d_vp.as<float>(), flip_all,
                 d_raw.as<float4>(), d_cloud_off.as<int64_t>(), d_nbr.as<int>(), d_nmom.as<double>(),
                 d_nsel.as<int>(), d_nwork.as<int>(), nrm.as<float4>(), s);
  prof.end(span, s, spans);
  has_nrm = true;
}

void CloudSet::build_near_mask(hipStream_t s, double r) {
  // dilation in cells: a point within r of a query lies at most ceil(r / h) + 1
  // cells away along each axis (the +1 covers positions inside the cells and
  // binning rounding)
  // (in double: the default radius, sqrt(DBL_MAX), spans more cells than an int
  // holds, and as one it passed for a small mask whose dilation took minutes)
  double kd_max = 0.0;
  for (const GridDesc& g : grids)
    if (g.npts > 0) kd_max = std::max(kd_max, ceil(r * 1.0001 * (double)g.inv_h) + 1.0);
  const bool use = std::isfinite(r) && r > 0.0 && kd_max <= kMaxNearCells && total_cells > 0;
  // the same word offsets launch_set_near gives the device copy
  int64_t words = 0;
  for (GridDesc& g : grids) {
    g.near_r = use ? (float)r : 0.0f;
    g.near_off = words;
    words += (int64_t)near_row_words(g.nx) * g.ny * g.nz;
  }
  launch_set_near(d_grids.as<GridDesc>(), n, use ? (float)r : 0.0f, s);
  if (use) {
    d_near.reserve((size_t)std::max<int64_t>(words, 1) * sizeof(uint32_t));
    d_near_tmp.reserve((size_t)std::max<int64_t>(words, 1) * sizeof(uint32_t));
    launch_near_mask(d_grids.as<GridDesc>(), n, d_cell_start.as<int>(), words, (float)r,
                     d_near.as<uint32_t>(), d_near_tmp.as<uint32_t>(), s);
  }
}

void CloudSet::normals_to_input_order(hipStream_t s, float* d_nrm3, float* d_curv) {
  launch_unsort_normals(d_pts.as<float4>(), d_nrm.as<float4>(), d_cloud_of_sorted.as<int>(),
                        d_cloud_off.as<int64_t>(), total_pts, total_raw, d_nrm3, d_curv, s);
}

// ------------------------------------------------------------------ engine

Engine::~Engine() { reset_graph(); }

// Never throws: also runs from the destructor.
void Engine::reset_graph() {
  eager_key_set_ = false;
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  if (tail_exec) (void)hipGraphExecDestroy(tail_exec);
  if (tail_graph) (void)hipGraphDestroy(tail_graph);
  if (split_exec) (void)hipGraphExecDestroy(split_exec);
  if (split_graph) (void)hipGraphDestroy(split_graph);
  exec = nullptr;
  graph = nullptr;
  tail_exec = nullptr;
  tail_graph = nullptr;
  split_exec = nullptr;
  split_graph = nullptr;
}

// Live 64-point tiles at or below which a chunk runs the four-lanes-per-query
// search: more fill the chip with one lane per query (a fresh 24-capture cycle's
// kernels, with the seeds' balls walked row by row: 7810 us at 2048, 7420 at 4096,
// 7520 at 8192, 7820 with the split in every launch); LCR_SPLIT_TILES (read at every
// setup) overrides it, 0 turns the split off.
static int icp_split_units() {
  const char* e = getenv("LCR_SPLIT_TILES");
  if (e && *e) return std::max(0, atoi(e));
  return 4096;
}

// The resident blocks of the search, fitness and split kernels per CU: properties
// of the code and the device type, queried once per kernel (a query takes tens of
// microseconds).
static int blocks_per_cu(int which, int tile, bool p2pl, int precision) {
  static std::mutex mu;
  static std::map<int, int> known;
  const int key = ((which * 4 + (tile == 64 ? 0 : (tile == 128 ? 1 : 2))) * 2 + (p2pl ? 1 : 0)) * 8 + precision;
  std::lock_guard<std::mutex> lock(mu);
  auto it = known.find(key);
  if (it != known.end()) return it->second;
  const int v = which >= 3   ? icp_split_blocks_per_cu(tile, p2pl, which == 4)
                : which == 2 ? fitness_max_blocks_per_cu(tile)
                             : icp_max_blocks_per_cu(tile, p2pl, precision, which != 0);
  known[key] = v;
  return v;
}

namespace {
// tile -> its instance (instances in tile order): the last whose first tile is <= t
__global__ void k_tile_pairs(const PairDesc* __restrict__ pairs, int npairs, int ntiles,
                             int* __restrict__ out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  int lo = 0, hi = npairs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pairs[mid].tile_begin <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  out[t] = lo;
}
}  // namespace

void Engine::setup(hipStream_t s, const CloudSet& cs, const std::vector<int>& src,
                   const std::vector<int>& tgt, const std::vector<double>& r2, int tile_pts) {
  reset_graph();
  matched = false;
  tile = (tile_pts == 64 || tile_pts == 128 || tile_pts == 256) ? tile_pts : 256;
  npairs = (int)src.size();
  hp.assign(npairs, PairDesc{});
  std::vector<int> gt;
  ntiles = 0;
  for (int p = 0; p < npairs; ++p) {
    PairDesc& d = hp[p];
    d.src = src[p];
    d.tgt = tgt[p];
    d.tile_begin = ntiles;
    d.ntiles = (cs.grids[d.src].npts + tile - 1) / tile;
    d.max_corr_d2 = r2[p];
    for (int t = 0; t < d.ntiles; t += gate_stride(d.ntiles)) gt.push_back(ntiles + t);
    ntiles += d.ntiles;
  }
  ngate_tiles = (int)gt.size();
  d_pairs.reserve(std::max(npairs, 1) * sizeof(PairDesc));
  d_tile_pair.reserve(std::max(ntiles, 1) * sizeof(int));
  d_state.reserve((size_t)(npairs + 1) * sizeof(PairState));
  d_partials.reserve((size_t)std::max(ntiles, 1) * kMaxVals * sizeof(double));
  d_prev.reserve((size_t)std::max(ntiles, 1) * tile * sizeof(int));
  d_guess.reserve((size_t)std::max(npairs, 1) * 16 * sizeof(double));
  h_state.reserve((size_t)(npairs + 1) * sizeof(PairState));
  h_guess.reserve((size_t)std::max(npairs, 1) * 16 * sizeof(double));
  // live-tile lists (each run compacts them first)
  d_it_list.reserve((size_t)std::max(ntiles, 1) * sizeof(int2));
  d_fit_list.reserve((size_t)std::max(ntiles, 1) * sizeof(int2));
  d_fit_order.reserve((size_t)std::max(ntiles, 1) * sizeof(int2));
  d_fit_flags.reserve((size_t)std::max(ntiles, 1) * sizeof(int));
  d_list_count.reserve(2 * sizeof(int));
  d_gate_tiles.reserve(std::max<size_t>(gt.size(), 1) * sizeof(int));
  if (!d_fetch.p) {
    d_fetch.reserve(kFetchCounters * sizeof(int));
    launch_fill_i32(d_fetch.as<int>(), kFetchCounters, 0, s);
  }
  // through pinned memory; every run ends with a wait for the stream, so the last
  // setup's copies are done before this one rewrites it
  const size_t pair_bytes = (size_t)npairs * sizeof(PairDesc);
  h_setup.reserve(pair_bytes + gt.size() * sizeof(int));
  if (npairs > 0) {
    memcpy(h_setup.p, hp.data(), pair_bytes);
    LCR_HIP(hipMemcpyAsync(d_pairs.p, h_setup.p, pair_bytes, hipMemcpyHostToDevice, s));
  }
  if (ngate_tiles > 0) {
    char* g = h_setup.as<char>() + pair_bytes;
    memcpy(g, gt.data(), gt.size() * sizeof(int));
    LCR_HIP(hipMemcpyAsync(d_gate_tiles.p, g, gt.size() * sizeof(int), hipMemcpyHostToDevice, s));
  }
  if (ntiles > 0)
    hipLaunchKernelGGL(k_tile_pairs, dim3((unsigned)((ntiles + 255) / 256)), dim3(256), 0, s,
                       d_pairs.as<PairDesc>(), npairs, ntiles, d_tile_pair.as<int>());
  const int cus = device_cu_count();
  setup_precision = c.precision;
  const bool pl = c.point_to_plane != 0;
  for (int ring = 0; ring < 2; ++ring) {
    int nb = std::min(std::max(ntiles, 1), cus * blocks_per_cu(ring, tile, pl, c.precision));
    nb = std::max(8, (nb + 7) / 8 * 8);
    (ring ? nblocks_ring : nblocks) = nb;
  }
  int nf = std::min(std::max(ntiles, 1), cus * blocks_per_cu(2, tile, false, 0));
  nblocks_fit = std::max(8, (nf + 7) / 8 * 8);
  split_units = icp_split_units();
  if (split_units > 0) {
    for (int ring = 0; ring < 2; ++ring) {
      int ns = std::min(std::max(std::min(ntiles, split_units / (tile / 64)), 1),
                        cus * blocks_per_cu(3 + ring, tile, pl, 0));
      ns = std::max(8, (ns + 7) / 8 * 8);
      (ring ? nblocks_split_ring : nblocks_split) = ns;
    }
  }
}

// LCR_FIT_ORDER=fixed: the fitness passes in fixed per-block shares of the tiles
// instead of tiles handed out by counters (read at every run).
static bool fitness_fixed_shares() {
  const char* e = getenv("LCR_FIT_ORDER");
  return e && strcmp(e, "fixed") == 0;
}

IcpBuffers Engine::buffers(const CloudSet& cs) const {
  IcpBuffers b;
  memset(&b, 0, sizeof b);  // padding takes part in the graph key comparison
  b.grids = cs.d_grids.as<GridDesc>();
  b.cell_start = cs.d_cell_start.as<int>();
  b.pts = cs.d_pts.as<float4>();
  b.nrm = cs.has_nrm ? cs.d_nrm.as<float4>() : nullptr;
  b.nodes = cs.d_nodes.as<float4>();
  b.tpts = cs.d_tpts.as<float4>();
  b.tpos = cs.d_tpos.as<int>();
  b.pairs = d_pairs.as<PairDesc>();
  b.tile_pair = d_tile_pair.as<int>();
  b.state = d_state.as<PairState>();
  b.partials = d_partials.as<double>();
  b.prev = d_prev.as<int>();
  b.near = cs.d_near.p ? cs.d_near.as<uint32_t>() : nullptr;
  b.gate_tiles = d_gate_tiles.as<int>();
  b.ngate_tiles = ngate_tiles;
  b.it_list = d_it_list.as<int2>();
  b.it_count = d_list_count.as<int>();
  b.fit_list = d_fit_list.as<int2>();
  b.fit_count = d_list_count.as<int>() + 1;
  b.fetch = fitness_fixed_shares() ? nullptr : d_fetch.as<int>();
  b.fit_order = b.fetch ? d_fit_order.as<int2>() : nullptr;
  b.fit_flags = d_fit_flags.as<int>();
  b.ntiles = ntiles;
  b.npairs = npairs;
  b.tile = tile;
  b.morton = (c.morton && cs.d_tpts.p) ? 1 : 0;
  return b;
}

// Waits until a kernel on `s` has set *flag (coherent host memory).  Ends in any
// case: once the stream has nothing left to run or reports an error.
static void wait_flag(const int* flag, hipStream_t s) {
  for (unsigned spins = 1;; ++spins) {
    if (__atomic_load_n(flag, __ATOMIC_ACQUIRE)) return;
    __builtin_ia32_pause();
    if (spins % 1024 != 0) continue;
    const hipError_t e = hipStreamQuery(s);
    if (e == hipErrorNotReady) continue;
    LCR_HIP(e);
    if (__atomic_load_n(flag, __ATOMIC_ACQUIRE)) return;
    throw Error{-2, "the iterations ended without their count"};
  }
}

// The run is: state init -> chunks of kChunk iterations -> fitness.  Each chunk
// ends with a count of still-active instances in host memory; the host stops
// launching chunks once it reads zero, so converged cycles do not replay
// empty iterations.  With the profiler off each chunk (and the tail) replays a
// captured hipGraph; HIP events recorded inside a captured graph cannot be timed
// afterwards, so with the profiler on the same launches are issued eagerly with
// an event pair around each kernel.
bool Engine::ring_only(const CloudSet& cs) const {
  if (c.precision != 0 || npairs == 0) return false;
  for (const PairDesc& d : hp) {
    // the same float arithmetic as nn_query's per-query test
    const float r = (float)sqrt(d.max_corr_d2);
    const float rlim = r * 1.00001f;
    if (!std::isfinite(r) || !(rlim * cs.grids[d.tgt].inv_h <= kRingOnlyCells)) return false;
  }
  return true;
}

void Engine::run(hipStream_t s, const CloudSet& cs, const double* guesses, bool use_graph,
                 const std::function<void()>& pre) {
  if (npairs == 0) return;
  matched = false;
  Profiler& prof = Profiler::get();
  c.ring_only = ring_only(cs) ? 1 : 0;
  const int nb_search = c.ring_only ? nblocks_ring : nblocks;
  const int nb_split = c.ring_only ? nblocks_split_ring : nblocks_split;
  const IcpBuffers b = buffers(cs);
  if (guesses) {
    memcpy(h_guess.p, guesses, (size_t)npairs * 16 * sizeof(double));
  } else {
    double* g = h_guess.as<double>();
    for (int p = 0; p < npairs; ++p)
      for (int i = 0; i < 16; ++i) g[16 * p + i] = (i % 5 == 0) ? 1.0 : 0.0;
  }
  LCR_HIP(hipMemcpyAsync(d_guess.p, h_guess.p, (size_t)npairs * 16 * sizeof(double),
                         hipMemcpyHostToDevice, s));
  if (pre) pre();
  launch_state_init(d_state.as<PairState>(), d_guess.as<double>(), d_pairs.as<PairDesc>(),
                    cs.d_grids.as<GridDesc>(), npairs, s);
  auto compact_all = [&] {
    launch_compact_tiles(b, d_it_list.as<int2>(), d_list_count.as<int>(), d_fit_list.as<int2>(),
                         d_list_count.as<int>() + 1, nullptr, s);
  };
  const bool gated = gate_h > 1 && ntiles > 0;
  if (!gated) compact_all();
  h_active.reserve(3 * sizeof(int));
  const bool split_ok = use_split();
  // A run of a new handle, or of other buffers or parameters than the last, issues
  // its launches directly; capturing and instantiating its three graphs (about half
  // a millisecond) waits until the same run comes again.
  bool eager = !use_graph || prof.on();
  if (!eager) {
    const GraphKey key = graph_key(b);
    const bool captured = exec && tail_exec && (!split_ok || split_exec) && key == graph_key_;
    eager = !captured && !(eager_key_set_ && key == eager_key_);
    eager_key_ = key;
    eager_key_set_ = true;
  }
  std::vector<Profiler::Span> spans;
  if (gated) {
    const int k = prof.begin("gate", s, &spans);
    // XCD-contiguous: the hypotheses of a pair share its target grid in one L2
    // (74 pairs x 15 hypotheses: 21.4 against 21.6 ms per cycle step in grid-stride
    // order)
    launch_fitness(b, 0.0, nblocks_fit, s, true, 0);
    launch_gate(d_state.as<PairState>(), npairs / gate_h, gate_h, s);
    compact_all();
    prof.end(k, s, &spans);
  }
  auto chunk = [&](std::vector<Profiler::Span>* sp, bool split) {
    for (int it = 0; it < kChunk; ++it) {
      // the split launches are also counted on their own
      const int k = prof.begin("icp_iteration", s, sp);
      const int ks = split ? prof.begin("icp_iteration_split", s, sp) : -1;
      if (split)
        launch_icp_search_split(b, c, nb_split, s);
      else
        launch_icp_search(b, c, nb_search, s);
      prof.end(ks, s, sp);
      prof.end(k, s, sp);
      const int k2 = prof.begin("icp_solve", s, sp);
      launch_icp_solve(b, c, s);
      prof.end(k2, s, sp);
    }
    launch_compact_tiles(b, d_it_list.as<int2>(), d_list_count.as<int>(), nullptr, nullptr,
                         h_active.as<int>(), s);
  };
  auto tail = [&](std::vector<Profiler::Span>* sp) {
    const int k = prof.begin("fitness", s, sp);
    // one launch over every instance (with fixed shares, XCD-contiguous tiles keep
    // each target's tree in one L2)
    launch_fitness(b, DBL_MAX, nblocks_fit, s, false, 0, fit_split());
    prof.end(k, s, sp);
    LCR_HIP(hipMemcpyAsync(h_state.p, d_state.p, (size_t)npairs * sizeof(PairState),
                           hipMemcpyDeviceToHost, s));
  };
  if (!eager) {
    const GraphKey key = graph_key(b);
    if (!exec || !tail_exec || (split_ok && !split_exec) || !(key == graph_key_)) {
      reset_graph();
      capture(s, [&] { chunk(nullptr, false); }, &graph, &exec);
      if (split_ok) capture(s, [&] { chunk(nullptr, true); }, &split_graph, &split_exec);
      capture(s, [&] { tail(nullptr); }, &tail_graph, &tail_exec);
      graph_key_ = key;
    }
  }
  // the first chunk splits when all of the tiles fit under split_units, later ones
  // when the previous chunk left that few live
  bool split = split_fits(ntiles);
  const int max_chunks = ntiles > 0 ? (c.max_iterations + kChunk - 1) / kChunk : 0;
  int* const host = h_active.as<int>();
  for (int k = 0; k < max_chunks; ++k) {
    host[2] = 0;  // the last chunk, if any, has set it
    if (eager)
      chunk(&spans, split);
    else
      LCR_HIP(hipGraphLaunch(split ? split_exec : exec, s));
    wait_flag(&host[2], s);
    if (host[0] == 0) break;
    split = split_fits(host[1]);
  }
  if (ntiles > 0) {
    if (eager)
      tail(&spans);
    else
      LCR_HIP(hipGraphLaunch(tail_exec, s));
  } else {
    LCR_HIP(hipMemcpyAsync(h_state.p, d_state.p, (size_t)npairs * sizeof(PairState),
                           hipMemcpyDeviceToHost, s));
  }
  LCR_HIP(hipStreamSynchronize(s));
  matched = true;
  if (!spans.empty()) prof.collect(spans, false);
}

void Engine::capture(hipStream_t s, const std::function<void()>& f, hipGraph_t* g,
                     hipGraphExec_t* e) {
  LCR_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  try {
    f();
  } catch (...) {
    hipGraph_t t = nullptr;
    (void)hipStreamEndCapture(s, &t);
    if (t) (void)hipGraphDestroy(t);
    throw;
  }
  LCR_HIP(hipStreamEndCapture(s, g));
  LCR_HIP(hipGraphInstantiate(e, *g, nullptr, nullptr, 0));
}

// Everything a captured graph bakes in: kernel arguments and buffer addresses.
Engine::GraphKey Engine::graph_key(const IcpBuffers& b) const {
  GraphKey k;
  memset(&k, 0, sizeof k);
  k.b = b;
  k.c = c;
  k.nblocks = c.ring_only ? nblocks_ring : nblocks;
  k.nblocks_fit = nblocks_fit;
  k.nblocks_split = use_split() ? (c.ring_only ? nblocks_split_ring : nblocks_split) : 0;
  k.guess = d_guess.p;
  k.hstate = h_state.p;
  k.hactive = h_active.p;
  return k;
}

void Engine::run_fitness(hipStream_t s, const CloudSet& cs, double max_range) {
  if (npairs == 0) return;
  Profiler& prof = Profiler::get();
  std::vector<Profiler::Span> spans;
  IcpBuffers b = buffers(cs);
  if (!matched) {  // other tiles since the last run: every tile, no seeds
    b.prev = nullptr;
    b.fit_list = nullptr;
    b.fit_count = nullptr;
  }
  if (ntiles > 0) {
    const int sp = prof.begin("fitness", s, &spans);
    launch_fitness(b, max_range, nblocks_fit, s, false, c.interleave, fit_split());
    prof.end(sp, s, &spans);
  }
  LCR_HIP(hipMemcpyAsync(h_state.p, d_state.p, (size_t)npairs * sizeof(PairState),
                         hipMemcpyDeviceToHost, s));
  LCR_HIP(hipStreamSynchronize(s));
  if (!spans.empty()) prof.collect(spans, false);
}

}  // namespace lcr
