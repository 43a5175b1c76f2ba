// proposal.cpp -- host side of the learned initial-pose proposal (K9): weights,
// device-resident training set, forward / backward / Adam on the GPU, and the
// per-pair inference the batched cycle uses as an extra pose hypothesis.
#include <float.h>
#include <math.h>
#include <string.h>

#include <algorithm>
#include <memory>
#include <random>
#include <vector>

#include "../../include/lcr.h"
#include "lcr_kernels.hpp"
#include "runtime.hpp"

namespace lcr {

namespace {

// ---- device helpers local to the proposal

// Inputs of the network for every pair of a cycle: n_out points subsampled evenly
// from each raw cloud, the source moved by the pair's seed T0, both normalised by
// the target sample's centroid and RMS radius.  k_prop_frame: one block per pair,
// its first kPrepKeep samples per thread loaded together and kept for both sums,
// which a fixed LDS tree folds, so the frame does not depend on timing.
// k_prop_inputs: a thread per sample.  A sample is a cache line of its own, so one
// block per pair for all of it waited on its CU's loads (36 pairs, 8192 samples:
// 64 us, now 28 + 9).
constexpr int kPrepThreads = 1024;

// Sample i of n_out taken evenly from a cloud of n > 0 points: floor(i * n / n_out),
// in 32-bit arithmetic when the product fits.
__device__ __forceinline__ int64_t sample_at(int i, int64_t n, int n_out) {
  if (n < ((int64_t)1 << 31) / n_out) return (int64_t)((unsigned)(i * (int)n) / (unsigned)n_out);
  return (int64_t)i * n / n_out;
}

template <int N>
__device__ __forceinline__ void prep_sum(double (&v)[N], double (*red)[N]) {
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < N; ++k) red[t][k] = v[k];
  __syncthreads();
  for (int o = kPrepThreads / 2; o > 0; o >>= 1) {
    if (t < o) {
#pragma unroll
      for (int k = 0; k < N; ++k) red[t][k] += red[t + o][k];
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = red[0][k];
  __syncthreads();  // red is reused
}

constexpr int kPrepKeep = 8;

__global__ void __launch_bounds__(kPrepThreads)
k_prop_frame(const float4* __restrict__ raw, const int64_t* __restrict__ cloud_off,
             const int* __restrict__ tgt, int n_out, double* __restrict__ norm,
             float* __restrict__ frame) {
  __shared__ double red[kPrepThreads][4];
  const int pr = blockIdx.x, t = threadIdx.x;
  const int64_t t0 = cloud_off[tgt[pr]], nt = cloud_off[tgt[pr] + 1] - t0;
  const int taken = nt > 0 ? n_out : 0;  // an empty cloud has nothing to read
  float4 keep[kPrepKeep];
#pragma unroll
  for (int u = 0; u < kPrepKeep; ++u) {
    const int i = t + u * kPrepThreads;
    keep[u] = i < taken ? raw[t0 + sample_at(i, nt, n_out)] : make_float4(NAN, NAN, NAN, NAN);
  }
  double a[4] = {0, 0, 0, 0};
  auto add = [&](const float4& q) {
    if (isfinite(q.x) && isfinite(q.y) && isfinite(q.z)) {
      a[0] += q.x;
      a[1] += q.y;
      a[2] += q.z;
      a[3] += 1.0;
    }
  };
#pragma unroll
  for (int u = 0; u < kPrepKeep; ++u) add(keep[u]);
  for (int i = t + kPrepKeep * kPrepThreads; i < taken; i += kPrepThreads)
    add(raw[t0 + sample_at(i, nt, n_out)]);
  prep_sum<4>(a, red);
  const double n = a[3] > 0 ? a[3] : 1.0;
  const double cx = a[0] / n, cy = a[1] / n, cz = a[2] / n;
  double b[2] = {0, 0};
  auto spread = [&](const float4& q) {
    if (isfinite(q.x) && isfinite(q.y) && isfinite(q.z)) {
      const double dx = q.x - cx, dy = q.y - cy, dz = q.z - cz;
      b[0] += dx * dx + dy * dy + dz * dz;
      b[1] += 1.0;
    }
  };
#pragma unroll
  for (int u = 0; u < kPrepKeep; ++u) spread(keep[u]);
  for (int i = t + kPrepKeep * kPrepThreads; i < taken; i += kPrepThreads)
    spread(raw[t0 + sample_at(i, nt, n_out)]);
  prep_sum<2>(b, reinterpret_cast<double(*)[2]>(red));
  const double rr = b[1] > 0 ? sqrt(b[0] / b[1]) : 1.0;
  const double rad = rr > 1e-12 ? rr : 1.0;
  if (t == 0) {
    frame[pr * 4 + 0] = (float)cx;
    frame[pr * 4 + 1] = (float)cy;
    frame[pr * 4 + 2] = (float)cz;
    frame[pr * 4 + 3] = (float)rad;
    norm[pr] = 1.0 / rad;
  }
}

// `per` blocks for a pair's target sample, then `per` for its source's.
__global__ void __launch_bounds__(256)
k_prop_inputs(const float4* __restrict__ raw, const int64_t* __restrict__ cloud_off,
              const int* __restrict__ src, const int* __restrict__ tgt,
              const double* __restrict__ guesses, int guess_stride, int n_out,
              const double* __restrict__ norm, const float* __restrict__ frame, int per,
              float4* __restrict__ X) {
  const int part = (int)blockIdx.x / per, pr = part >> 1;
  const int i = ((int)blockIdx.x % per) * 256 + (int)threadIdx.x;
  if (i >= n_out) return;
  const bool source = part & 1;
  const int cloud = source ? src[pr] : tgt[pr];
  const int64_t o = cloud_off[cloud], n = cloud_off[cloud + 1] - o;
  const float inv = (float)norm[pr];
  const float c0 = frame[pr * 4], c1 = frame[pr * 4 + 1], c2 = frame[pr * 4 + 2];
  float4* out = X + (int64_t)pr * 2 * n_out + (source ? 0 : n_out);
  const float4 p = n > 0 ? raw[o + sample_at(i, n, n_out)] : make_float4(NAN, NAN, NAN, NAN);
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (isfinite(p.x) && isfinite(p.y) && isfinite(p.z)) {
    float m[3] = {p.x, p.y, p.z};
    if (source) {
      const double* T = guesses + (int64_t)pr * guess_stride * 16;
#pragma unroll
      for (int r = 0; r < 3; ++r)
        m[r] = (float)(T[4 * r] * p.x + T[4 * r + 1] * p.y + T[4 * r + 2] * p.z + T[4 * r + 3]);
    }
    v = make_float4((m[0] - c0) * inv, (m[1] - c1) * inv, (m[2] - c2) * inv, 0.f);
  }
  out[i] = v;
}

// learned guess = [R(omega) | s tau + c - R c] * T0, written to the pair's learned slot
__global__ void k_prop_guess(const float* __restrict__ out, const float* __restrict__ frame,
                             int npairs, int guess_stride, int slot, double* __restrict__ guesses) {
  const int pr = blockIdx.x * blockDim.x + threadIdx.x;
  if (pr >= npairs) return;
  const double w0 = out[pr * 6], w1 = out[pr * 6 + 1], w2 = out[pr * 6 + 2];
  const double th = sqrt(w0 * w0 + w1 * w1 + w2 * w2);
  double R[9];
  if (th < 1e-12) {
    for (int i = 0; i < 9; ++i) R[i] = (i % 4 == 0) ? 1.0 : 0.0;
  } else {
    const double kx = w0 / th, ky = w1 / th, kz = w2 / th, s = sin(th), c = cos(th), v = 1.0 - c;
    R[0] = c + kx * kx * v;
    R[1] = kx * ky * v - kz * s;
    R[2] = kx * kz * v + ky * s;
    R[3] = ky * kx * v + kz * s;
    R[4] = c + ky * ky * v;
    R[5] = ky * kz * v - kx * s;
    R[6] = kz * kx * v - ky * s;
    R[7] = kz * ky * v + kx * s;
    R[8] = c + kz * kz * v;
  }
  const double cx = frame[pr * 4], cy = frame[pr * 4 + 1], cz = frame[pr * 4 + 2], sg = frame[pr * 4 + 3];
  double D[16];
  for (int r = 0; r < 3; ++r) {
    for (int k = 0; k < 3; ++k) D[4 * r + k] = R[3 * r + k];
    D[4 * r + 3] = sg * out[pr * 6 + 3 + r] + (r == 0 ? cx : (r == 1 ? cy : cz)) -
                   (R[3 * r] * cx + R[3 * r + 1] * cy + R[3 * r + 2] * cz);
  }
  D[12] = D[13] = D[14] = 0.0;
  D[15] = 1.0;
  const double* T0 = guesses + (int64_t)pr * guess_stride * 16;
  double* G = guesses + ((int64_t)pr * guess_stride + slot) * 16;
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) {
      double s = 0.0;
      for (int k = 0; k < 4; ++k) s += D[4 * i + k] * T0[4 * k + j];
      G[4 * i + j] = s;
    }
}

}  // namespace

struct ProposalImpl {
  int device = 0;
  Stream stream;
  const hipStream_t s;
  int cap_pairs = 0, cap_pts = 0;
  int step = 0;
  DevBuf W, M, V, G, W2t, W3t;
  DevBuf X, part_max, part_arg, F, ARG, Z, OUT, DOUT, loss_part, DZ, DG, part_grad, lab, losses, frame, norm;
  DevBuf ds_X, ds_lab;
  int ds_pairs = 0, ds_pts = 0;
  HostBuf h_io;

  static int current_device() {
    int d = 0;
    LCR_HIP(hipGetDevice(&d));
    return d;
  }
  ProposalImpl() : device(current_device()), stream(device), s(stream.s) {
    W.reserve(kEncNParam * sizeof(float));
    M.reserve(kEncNParam * sizeof(float));
    V.reserve(kEncNParam * sizeof(float));
    G.reserve(kEncNParam * sizeof(float));
    W2t.reserve(64 * 128 * sizeof(__bf16));
    W3t.reserve(128 * 256 * sizeof(__bf16));
    // no block is clear when it is taken
    LCR_HIP(hipMemsetAsync(W.p, 0, kEncNParam * sizeof(float), s));
    LCR_HIP(hipMemsetAsync(W2t.p, 0, 64 * 128 * sizeof(__bf16), s));
    LCR_HIP(hipMemsetAsync(W3t.p, 0, 128 * 256 * sizeof(__bf16), s));
    reset_optimizer();
    LCR_HIP(hipStreamSynchronize(s));  // a cycle reads the weights on its own stream
  }
  ~ProposalImpl() { (void)stream.idle(); }  // before the buffers go back to the pool
  void bind() const { LCR_HIP(hipSetDevice(device)); }
  void reset_optimizer() {
    LCR_HIP(hipMemsetAsync(M.p, 0, kEncNParam * sizeof(float), s));
    LCR_HIP(hipMemsetAsync(V.p, 0, kEncNParam * sizeof(float), s));
    step = 0;
  }
  void reserve(int npairs, int npts) {
    if (npairs <= cap_pairs && npts <= cap_pts) return;
    const int64_t P = std::max(cap_pairs, npairs), C = 2 * P, N = std::max(cap_pts, npts);
    cap_pairs = cap_pts = 0;  // until every buffer is there
    const int64_t chunks = enc_forward_chunks((int)N);
    part_max.reserve(C * chunks * 256 * sizeof(float));
    part_arg.reserve(C * chunks * 256 * sizeof(int));
    F.reserve(C * 256 * sizeof(float));
    ARG.reserve(C * 256 * sizeof(int));
    Z.reserve(P * 256 * sizeof(float));
    OUT.reserve(P * 6 * sizeof(float));
    DOUT.reserve(P * 6 * sizeof(float));
    loss_part.reserve(P * 6 * sizeof(float));
    DZ.reserve(P * 256 * sizeof(float));
    DG.reserve(P * 512 * sizeof(float));
    part_grad.reserve(enc_part_grad_floats((int)P) * sizeof(float));
    lab.reserve(P * 6 * sizeof(float));
    cap_pairs = (int)P;
    cap_pts = (int)N;
  }
  // the batch's own points (training and prediction read the resident set in place)
  void reserve_points(int npairs, int npts) {
    X.reserve((size_t)2 * npairs * npts * sizeof(float4));
  }
  EncBuffers bufs() const {
    EncBuffers e;
    e.X = X.as<float4>();
    e.sel = nullptr;
    e.W = W.as<float>();
    e.W2t = W2t.as<__bf16>();
    e.W3t = W3t.as<__bf16>();
    e.part_max = part_max.as<float>();
    e.part_arg = part_arg.as<int>();
    e.F = F.as<float>();
    e.ARG = ARG.as<int>();
    e.Z = Z.as<float>();
    e.OUT = OUT.as<float>();
    e.DOUT = DOUT.as<float>();
    e.loss_part = loss_part.as<float>();
    e.DZ = DZ.as<float>();
    e.DG = DG.as<float>();
    e.part_grad = part_grad.as<float>();
    e.G = G.as<float>();
    return e;
  }
  // host clouds (npairs * npts * 3 floats each) -> X as (src0, tgt0, src1, tgt1, ...)
  void upload_pairs(const float* src, const float* tgt, int npairs, int npts) {
    reserve(npairs, npts);
    reserve_points(npairs, npts);
    const int64_t n = (int64_t)npairs * 2 * npts;
    h_io.reserve((size_t)n * sizeof(float4));
    float4* h = h_io.as<float4>();
    for (int b = 0; b < npairs; ++b)
      for (int side = 0; side < 2; ++side) {
        const float* in = (side == 0 ? src : tgt) + (int64_t)b * npts * 3;
        float4* o = h + ((int64_t)b * 2 + side) * npts;
        for (int p = 0; p < npts; ++p) o[p] = make_float4(in[3 * p], in[3 * p + 1], in[3 * p + 2], 0.f);
      }
    LCR_HIP(hipMemcpyAsync(X.p, h, (size_t)n * sizeof(float4), hipMemcpyHostToDevice, s));
    LCR_HIP(hipStreamSynchronize(s));
  }
};

// Runs the network on every pair of a cycle (on the cycle's stream) and writes each
// pair's learned guess into its slot `slot` of the instance guesses (instances
// are pair-major with `stride` slots; slot 0 holds the plain seed).
void proposal_guesses(ProposalImpl& P, hipStream_t s, const CloudSet& cs, const int* d_src,
                      const int* d_tgt, int npairs, int npts, double* d_guess, int stride, int slot) {
  P.reserve(npairs, npts);
  P.reserve_points(npairs, npts);
  P.frame.reserve((size_t)npairs * 4 * sizeof(float));
  P.norm.reserve((size_t)npairs * sizeof(double));
  hipLaunchKernelGGL(k_prop_frame, dim3(npairs), dim3(kPrepThreads), 0, s, cs.d_raw.as<float4>(),
                     cs.d_cloud_off.as<int64_t>(), d_tgt, npts, P.norm.as<double>(),
                     P.frame.as<float>());
  const int per = (npts + 255) / 256;
  hipLaunchKernelGGL(k_prop_inputs, dim3((unsigned)npairs * 2 * per), dim3(256), 0, s,
                     cs.d_raw.as<float4>(), cs.d_cloud_off.as<int64_t>(), d_src, d_tgt, d_guess, stride,
                     npts, P.norm.as<double>(), P.frame.as<float>(), per, P.X.as<float4>());
  launch_enc_forward(P.bufs(), npairs, npts, nullptr, s);
  hipLaunchKernelGGL(k_prop_guess, dim3((npairs + 63) / 64), dim3(64), 0, s, P.OUT.as<float>(),
                     P.frame.as<float>(), npairs, stride, slot, d_guess);
}

}  // namespace lcr

using namespace lcr;

struct lcr_proposal {
  ProposalImpl impl;
};

lcr::ProposalImpl* lcr::proposal_impl(lcr_proposal* p) { return p ? &p->impl : nullptr; }

static inline int lcr_set_error_(int code, const char* msg) { return set_last_error(code, msg); }

template <class F>
static int pguard(F&& f) {
  try {
    return f();
  } catch (const Error& e) {
    return lcr_set_error_(e.code, e.msg.c_str());
  } catch (const std::bad_alloc&) {
    return lcr_set_error_(LCR_E_HIP, "out of memory");
  }
}

extern "C" {

int lcr_proposal_create(lcr_proposal** out) {
  return pguard([&]() -> int {
    if (!out) return lcr_set_error_(LCR_E_ARG, "out is NULL");
    *out = new lcr_proposal();
    return LCR_OK;
  });
}

void lcr_proposal_destroy(lcr_proposal* p) {
  if (!p) return;
  try {
    p->impl.bind();
  } catch (...) {
  }
  delete p;
}

int lcr_proposal_set_weights(lcr_proposal* p, const float* w, int64_t n) {
  return pguard([&]() -> int {
    if (!p || !w || n != kEncNParam) return lcr_set_error_(LCR_E_ARG, "expected 174470 weights");
    ProposalImpl& P = p->impl;
    P.bind();
    LCR_HIP(hipMemcpyAsync(P.W.p, w, n * sizeof(float), hipMemcpyHostToDevice, P.s));
    launch_enc_bf16_weights(P.W.as<float>(), P.W2t.as<__bf16>(), P.W3t.as<__bf16>(), P.s);
    P.reset_optimizer();
    LCR_HIP(hipStreamSynchronize(P.s));
    return LCR_OK;
  });
}

int lcr_proposal_get_weights(lcr_proposal* p, float* w, int64_t n) {
  return pguard([&]() -> int {
    if (!p || !w || n != kEncNParam) return lcr_set_error_(LCR_E_ARG, "expected 174470 weights");
    ProposalImpl& P = p->impl;
    P.bind();
    LCR_HIP(hipMemcpyAsync(w, P.W.p, n * sizeof(float), hipMemcpyDeviceToHost, P.s));
    LCR_HIP(hipStreamSynchronize(P.s));
    return LCR_OK;
  });
}

int lcr_proposal_forward(lcr_proposal* p, const float* src, const float* tgt, int32_t n_pairs,
                         int32_t n_points, float* out) {
  return pguard([&]() -> int {
    if (!p || !src || !tgt || !out || n_pairs < 1 || n_points < 1)
      return lcr_set_error_(LCR_E_ARG, "invalid arguments");
    ProposalImpl& P = p->impl;
    P.bind();
    P.upload_pairs(src, tgt, n_pairs, n_points);
    launch_enc_forward(P.bufs(), n_pairs, n_points, nullptr, P.s);
    LCR_HIP(hipMemcpyAsync(out, P.OUT.p, (size_t)n_pairs * 6 * sizeof(float), hipMemcpyDeviceToHost,
                           P.s));
    LCR_HIP(hipStreamSynchronize(P.s));
    return LCR_OK;
  });
}

int lcr_proposal_loss_grad(lcr_proposal* p, const float* src, const float* tgt, const float* labels,
                           int32_t n_pairs, int32_t n_points, float* loss, float* grad) {
  return pguard([&]() -> int {
    if (!p || !src || !tgt || !labels || n_pairs < 1 || n_points < 1)
      return lcr_set_error_(LCR_E_ARG, "invalid arguments");
    ProposalImpl& P = p->impl;
    P.bind();
    P.upload_pairs(src, tgt, n_pairs, n_points);
    LCR_HIP(hipMemcpyAsync(P.lab.p, labels, (size_t)n_pairs * 6 * sizeof(float),
                           hipMemcpyHostToDevice, P.s));
    const EncBuffers e = P.bufs();
    launch_enc_forward(e, n_pairs, n_points, P.lab.as<float>(), P.s);
    launch_enc_backward(e, n_pairs, n_points, P.s);
    std::vector<float> lp((size_t)n_pairs * 6);
    LCR_HIP(hipMemcpyAsync(lp.data(), P.loss_part.p, lp.size() * sizeof(float),
                           hipMemcpyDeviceToHost, P.s));
    if (grad)
      LCR_HIP(hipMemcpyAsync(grad, P.G.p, kEncNParam * sizeof(float), hipMemcpyDeviceToHost, P.s));
    LCR_HIP(hipStreamSynchronize(P.s));
    if (loss) {
      double s = 0.0;
      for (float v : lp) s += v;
      *loss = (float)s;
    }
    return LCR_OK;
  });
}

int lcr_proposal_dataset(lcr_proposal* p, const float* src, const float* tgt, const float* labels,
                         int32_t n_pairs, int32_t n_points) {
  return pguard([&]() -> int {
    if (!p || !src || !tgt || !labels || n_pairs < 1 || n_points < 1)
      return lcr_set_error_(LCR_E_ARG, "invalid arguments");
    ProposalImpl& P = p->impl;
    P.bind();
    const int64_t per = 2 * (int64_t)n_points;
    P.ds_pairs = 0;  // no set until it is there
    P.ds_X.reserve((size_t)n_pairs * per * sizeof(float4));
    P.ds_lab.reserve((size_t)n_pairs * 6 * sizeof(float));
    // upload in slices through the pinned staging buffer
    const int slice = std::max(1, (int)std::min<int64_t>(n_pairs, (256ll << 20) / (per * 16)));
    std::vector<float4> tmp;
    for (int b0 = 0; b0 < n_pairs; b0 += slice) {
      const int nb = std::min(slice, n_pairs - b0);
      P.h_io.reserve((size_t)nb * per * sizeof(float4));
      float4* h = P.h_io.as<float4>();
      for (int b = 0; b < nb; ++b)
        for (int side = 0; side < 2; ++side) {
          const float* in = (side == 0 ? src : tgt) + (int64_t)(b0 + b) * n_points * 3;
          float4* o = h + ((int64_t)b * 2 + side) * n_points;
          for (int q = 0; q < n_points; ++q)
            o[q] = make_float4(in[3 * q], in[3 * q + 1], in[3 * q + 2], 0.f);
        }
      LCR_HIP(hipMemcpyAsync(P.ds_X.as<float4>() + (int64_t)b0 * per, h, (size_t)nb * per * 16,
                             hipMemcpyHostToDevice, P.s));
      LCR_HIP(hipStreamSynchronize(P.s));
    }
    LCR_HIP(hipMemcpyAsync(P.ds_lab.p, labels, (size_t)n_pairs * 6 * sizeof(float),
                           hipMemcpyHostToDevice, P.s));
    LCR_HIP(hipStreamSynchronize(P.s));
    P.ds_pairs = n_pairs;
    P.ds_pts = n_points;
    return LCR_OK;
  });
}

int lcr_proposal_synthesize(lcr_proposal* p, const float* shapes, const float* weights,
                            const double* perturb, int32_t n_pairs, int32_t n_points, float noise,
                            uint64_t seed, float* raw, float* frame) {
  return pguard([&]() -> int {
    if (!p || !shapes || !weights || !perturb || n_pairs < 1 || n_points < 1)
      return lcr_set_error_(LCR_E_ARG, "invalid arguments");
    ProposalImpl& P = p->impl;
    P.bind();
    const int64_t per = 2 * (int64_t)n_points;
    P.ds_pairs = 0;  // no set until it is there
    P.ds_X.reserve((size_t)n_pairs * per * sizeof(float4));
    P.ds_lab.reserve((size_t)n_pairs * 6 * sizeof(float));
    std::vector<double> Pinv((size_t)n_pairs * 16);
    for (int b = 0; b < n_pairs; ++b) {
      const double* M = perturb + 16 * (int64_t)b;
      double* I = &Pinv[16 * (size_t)b];
      for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 3; ++c) I[4 * r + c] = M[4 * c + r];  // R^T
      for (int r = 0; r < 3; ++r)
        I[4 * r + 3] = -(I[4 * r] * M[3] + I[4 * r + 1] * M[7] + I[4 * r + 2] * M[11]);
      I[12] = I[13] = I[14] = 0.0;
      I[15] = 1.0;
    }
    DevBuf d_shapes, d_w, d_P, d_Pi, d_raw, d_frame;
    d_shapes.reserve((size_t)n_pairs * 45 * sizeof(float));
    d_w.reserve((size_t)n_pairs * 3 * sizeof(float));
    d_P.reserve((size_t)n_pairs * 16 * sizeof(double));
    d_Pi.reserve((size_t)n_pairs * 16 * sizeof(double));
    LCR_HIP(hipMemcpyAsync(d_shapes.p, shapes, (size_t)n_pairs * 45 * 4, hipMemcpyHostToDevice, P.s));
    LCR_HIP(hipMemcpyAsync(d_w.p, weights, (size_t)n_pairs * 3 * 4, hipMemcpyHostToDevice, P.s));
    LCR_HIP(hipMemcpyAsync(d_P.p, perturb, (size_t)n_pairs * 16 * 8, hipMemcpyHostToDevice, P.s));
    LCR_HIP(hipMemcpyAsync(d_Pi.p, Pinv.data(), (size_t)n_pairs * 16 * 8, hipMemcpyHostToDevice, P.s));
    if (raw) d_raw.reserve((size_t)n_pairs * per * 3 * sizeof(float));
    if (frame) d_frame.reserve((size_t)n_pairs * 4 * sizeof(float));
    launch_synth_pairs(d_shapes.as<float>(), d_w.as<float>(), d_P.as<double>(), d_Pi.as<double>(),
                       n_pairs, n_points, noise, seed, P.ds_X.as<float4>(), P.ds_lab.as<float>(),
                       raw ? d_raw.as<float>() : nullptr, frame ? d_frame.as<float>() : nullptr, P.s);
    if (raw)
      LCR_HIP(hipMemcpyAsync(raw, d_raw.p, (size_t)n_pairs * per * 3 * 4, hipMemcpyDeviceToHost, P.s));
    if (frame)
      LCR_HIP(hipMemcpyAsync(frame, d_frame.p, (size_t)n_pairs * 4 * 4, hipMemcpyDeviceToHost, P.s));
    LCR_HIP(hipStreamSynchronize(P.s));
    P.ds_pairs = n_pairs;
    P.ds_pts = n_points;
    return LCR_OK;
  });
}

int lcr_proposal_predict(lcr_proposal* p, int32_t first, int32_t count, float* out, float* labels) {
  return pguard([&]() -> int {
    if (!p || !out || count < 1 || first < 0) return lcr_set_error_(LCR_E_ARG, "invalid arguments");
    ProposalImpl& P = p->impl;
    if (count > P.ds_pairs - first) return lcr_set_error_(LCR_E_ARG, "range beyond the resident set");
    P.bind();
    const int chunk = 512;
    for (int b0 = 0; b0 < count; b0 += chunk) {
      const int nb = std::min(chunk, count - b0);
      P.reserve(nb, P.ds_pts);
      EncBuffers e = P.bufs();
      e.X = P.ds_X.as<float4>() + (int64_t)(first + b0) * 2 * P.ds_pts;
      launch_enc_forward(e, nb, P.ds_pts, nullptr, P.s);
      LCR_HIP(hipMemcpyAsync(out + (int64_t)b0 * 6, P.OUT.p, (size_t)nb * 6 * 4, hipMemcpyDeviceToHost, P.s));
      if (labels)
        LCR_HIP(hipMemcpyAsync(labels + (int64_t)b0 * 6, P.ds_lab.as<float>() + (int64_t)(first + b0) * 6,
                               (size_t)nb * 6 * 4, hipMemcpyDeviceToHost, P.s));
      LCR_HIP(hipStreamSynchronize(P.s));
    }
    return LCR_OK;
  });
}

int lcr_proposal_train(lcr_proposal* p, int32_t steps, int32_t batch, float lr, uint64_t seed,
                       float* losses) {
  return pguard([&]() -> int {
    if (!p || steps < 1 || batch < 1) return lcr_set_error_(LCR_E_ARG, "invalid arguments");
    ProposalImpl& P = p->impl;
    if (P.ds_pairs < 1) return lcr_set_error_(LCR_E_STATE, "no training set");
    P.bind();
    batch = std::min(batch, P.ds_pairs);
    P.reserve(batch, P.ds_pts);
    P.losses.reserve((size_t)steps * sizeof(float));
    std::mt19937_64 rng(seed);
    std::vector<int> all((size_t)steps * batch);
    std::vector<int> perm(P.ds_pairs);
    for (int i = 0; i < P.ds_pairs; ++i) perm[i] = i;
    size_t pos = perm.size();
    for (auto& v : all) {
      if (pos == perm.size()) {
        std::shuffle(perm.begin(), perm.end(), rng);
        pos = 0;
      }
      v = perm[pos++];
    }
    DevBuf d_all;
    d_all.reserve(all.size() * sizeof(int));
    LCR_HIP(hipMemcpyAsync(d_all.p, all.data(), all.size() * sizeof(int), hipMemcpyHostToDevice,
                           P.s));
    EncBuffers e = P.bufs();
    e.X = P.ds_X.as<float4>();
    for (int st = 0; st < steps; ++st) {
      e.sel = d_all.as<int>() + (int64_t)st * batch;
      launch_enc_forward(e, batch, P.ds_pts, P.ds_lab.as<float>(), P.s);
      launch_enc_backward(e, batch, P.ds_pts, P.s);
      P.step += 1;
      launch_adam(e, P.M.as<float>(), P.V.as<float>(), batch, lr, P.step, P.losses.as<float>() + st, P.s);
    }
    if (losses)
      LCR_HIP(hipMemcpyAsync(losses, P.losses.p, (size_t)steps * sizeof(float), hipMemcpyDeviceToHost,
                             P.s));
    LCR_HIP(hipStreamSynchronize(P.s));
    return LCR_OK;
  });
}

}  // extern "C"
