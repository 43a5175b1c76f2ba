// encoder.hip -- K9: the learned initial-pose proposal (Siamese point encoder).
//
// No counterpart in the reference: the network takes the role of the coarse
// alignment that precedes fine registration (Super4PCS, scripts/alignment.sh:107).
// Per point 3 -> 64 -> 128 -> 256 (ReLU), max-pool per cloud, head 512 -> 256 -> 6
// (axis-angle, translation).  Layer 1 and the head run in FP32; layers 2 and 3 run
// on BF16 MFMA (v_mfma_f32_16x16x32_bf16) with FP32 accumulation, from BF16 copies
// of W2/W3 and BF16 activations h1/h2.
//
// Forward (k_enc_points): one block per cloud and up to kMaxPasses passes of kRows
// (128) points.  Layer 1 writes h1 (bf16) to LDS; each of the 4 waves computes 32
// channels of layer 2 for all rows (its weight fragments stay in registers) and
// writes h2 (bf16) to LDS, four channels per store; each wave then computes 64
// channels of layer 3 and folds bias, ReLU and the max-pool (with the lowest point
// index on ties) into registers, so only 256 (max, argmax) pairs per block leave
// the chip.  At 128 rows a block holds 53 KB of LDS and three blocks share a CU, so
// one block's MFMA work overlaps another's vector work.  Bound by the vector
// instructions around the MFMAs (per value of layer 3: bias, compare, select, max).
// 256 pairs x 8192 points: 682 -> 347 us (0.99 PFLOP/s; a large bf16 matrix product
// reaches 1.18 here) from one pass per block, weights loaded each time, two-byte
// stores of h2 and a bounds test per value.
//
// Backward: the max-pool sends each channel's gradient to one point, so the
// per-point layers only need the <= 256 argmax rows per cloud (k_enc_grad
// recomputes their activations and keeps the weight gradients' partial sums in
// registers).  Every sum is deterministic (fixed-order partials).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "lcr_kernels.hpp"

namespace lcr {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 128;      // points per forward pass (three blocks' LDS fit a CU)
constexpr int kMaxPasses = 8;   // passes per forward block at most
constexpr int kH1S = 64 + 8;    // LDS row strides (bf16), padded
constexpr int kH2S = 128 + 8;

__device__ __forceinline__ float relu(float v) { return v > 0.f ? v : 0.f; }

// The points of the batch's cloud c: clouds lie in X in batch order, or (sel: the
// pairs of a resident set that make up the batch) at their pair's place in the set.
__device__ __forceinline__ const float4* cloud_points(const float4* X, const int* sel, int cloud,
                                                      int npts) {
  const int64_t c = sel ? 2 * (int64_t)sel[cloud >> 1] + (cloud & 1) : cloud;
  return X + c * npts;
}

// ------------------------------------------------------------------ forward

// A block's points per pass; it runs `iters` passes over consecutive points, so the
// weight fragments are loaded once and one (max, argmax) pair per channel leaves
// per kRows * iters points.
__global__ void __launch_bounds__(256, 3)
k_enc_points(const float4* __restrict__ X, const int* __restrict__ sel, int npts, int iters,
             const float* __restrict__ W,
             const __bf16* __restrict__ W2t, const __bf16* __restrict__ W3t,
             float* __restrict__ part_max, int* __restrict__ part_arg) {
  __shared__ __attribute__((aligned(16))) __bf16 H1[kRows * kH1S];
  __shared__ __attribute__((aligned(16))) __bf16 H2[kRows * kH2S];
  static_assert(kRows == 128, "row and argmax arithmetic below");
  const int cloud = blockIdx.y, chunk = blockIdx.x, nchunks = gridDim.x;
  const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int l16 = lane & 15, q = lane >> 4, kq = q * 8;  // fragment row/col and k offset
  const float* W1 = W + kEncW1;
  const float* b1 = W + kEncB1;
  const int first = chunk * iters * kRows;
  const float4* Xc = cloud_points(X, sel, cloud, npts);
  bf16x8 w2[2][2], w3[4][4];
  f32x4 b2[2];
  float b3[4], best[4];
  int bidx[4];
#pragma unroll
  for (int jt = 0; jt < 2; ++jt) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      w2[jt][ks] = *(const bf16x8*)(W2t + (32 * w + 16 * jt + l16) * 64 + 32 * ks + kq);
    b2[jt] = *(const f32x4*)(W + kEncB2 + 32 * w + 16 * jt + 4 * q);
  }
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      w3[ct][ks] = *(const bf16x8*)(W3t + (64 * w + 16 * ct + l16) * 128 + 32 * ks + kq);
    b3[ct] = W[kEncB3 + 64 * w + 16 * ct + l16];
    // a maximum of at most 0 pools to 0 (ReLU) at no point, so only v > 0 matters
    best[ct] = 0.f;
    bidx[ct] = -1;
  }
  // points past the end repeat the last one: a repeat never beats its original,
  // which has the lower index
  const int row = t & (kRows - 1), j0 = (w >> 1) * 32;
  float4 x = Xc[min(first + row, npts - 1)];
  for (int it = 0; it < iters && first + it * kRows < npts; ++it) {
    // layer 1 (FP32), two threads per point, 32 outputs each
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x8 h;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int j = j0 + 8 * g + u;
        float a = b1[j];
        a = fmaf(x.x, W1[j], a);
        a = fmaf(x.y, W1[64 + j], a);
        a = fmaf(x.z, W1[128 + j], a);
        h[u] = (__bf16)fmaxf(a, 0.f);
      }
      *(bf16x8*)(H1 + row * kH1S + j0 + 8 * g) = h;
    }
    x = Xc[min(first + (it + 1) * kRows + row, npts - 1)];  // the next pass's point
    __syncthreads();
    // layer 2, transposed: wave w -> channels [32w, 32w + 32), a lane holds four
    // consecutive channels of one point and writes them together
#pragma unroll 2
    for (int rt = 0; rt < kRows / 16; ++rt) {
      f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16x8 hf = *(const bf16x8*)(H1 + (16 * rt + l16) * kH1S + 32 * ks + kq);
#pragma unroll
        for (int jt = 0; jt < 2; ++jt)
          acc[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w2[jt][ks], hf, acc[jt], 0, 0, 0);
      }
#pragma unroll
      for (int jt = 0; jt < 2; ++jt) {
        bf16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = (__bf16)fmaxf(acc[jt][e] + b2[jt][e], 0.f);
        *(bf16x4*)(H2 + (16 * rt + l16) * kH2S + 32 * w + 16 * jt + 4 * q) = h;
      }
    }
    __syncthreads();
    // layer 3 + bias + ReLU + max-pool: wave w -> channels [64w, 64w + 64)
#pragma unroll 2
    for (int rt = 0; rt < kRows / 16; ++rt) {
      f32x4 acc[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f},
                      {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 af = *(const bf16x8*)(H2 + (16 * rt + l16) * kH2S + 32 * ks + kq);
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, w3[ct][ks], acc[ct], 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int idx = (it * (kRows / 16) + rt) * 4 + e;  // wave-uniform
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          const float v = acc[ct][e] + b3[ct];
          bidx[ct] = v > best[ct] ? idx : bidx[ct];
          best[ct] = fmaxf(best[ct], v);
        }
      }
    }
  }
  // combine the 4 lane groups holding the same column (lanes l, l^16, l^32, l^48)
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    // point = 128 * pass + 16 * rt + 4 * q + e
    int p = bidx[ct] < 0 ? 0x7fffffff
                         : first + (bidx[ct] >> 5) * kRows + ((bidx[ct] >> 2) & 7) * 16 + 4 * q +
                               (bidx[ct] & 3);
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
      const float ov = __shfl_xor(best[ct], off, 64);
      const int op = __shfl_xor(p, off, 64);
      if (ov > best[ct] || (ov == best[ct] && op < p)) {
        best[ct] = ov;
        p = op;
      }
    }
    if (lane < 16) {
      const int64_t o = ((int64_t)cloud * nchunks + chunk) * 256 + 64 * w + 16 * ct + lane;
      part_max[o] = best[ct];
      part_arg[o] = p;
    }
  }
}

// fold chunk partials: feature F[cloud][c] and its point ARG[cloud][c]
__global__ void k_enc_pool(const float* __restrict__ part_max, const int* __restrict__ part_arg,
                           int nchunks, float* __restrict__ F, int* __restrict__ ARG) {
  const int cloud = blockIdx.x, c = threadIdx.x;
  float best = -1.f;
  int arg = 0;
  // eight chunks' loads in flight, the last one repeated to fill up (64 chunks: one
  // after the other 21 us, now 5.6)
  for (int k0 = 0; k0 < nchunks; k0 += 8) {
    float v[8];
    int a[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t o = ((int64_t)cloud * nchunks + min(k0 + u, nchunks - 1)) * 256 + c;
      v[u] = part_max[o];
      a[u] = part_arg[o];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      // chunks in point order: the first maximum keeps the lowest index
      arg = v[u] > best ? a[u] : arg;
      best = v[u] > best ? v[u] : best;
    }
  }
  F[cloud * 256 + c] = best < 0.f ? 0.f : best;
  ARG[cloud * 256 + c] = arg == 0x7fffffff ? 0 : arg;
}

// head: one block (256 threads) per pair; with labels (of pair sel[b] when given)
// also the loss and its gradient down to the hidden layer: dOut, dZ[j] = relu'(z)
// sum_o dOut[o] Hw2[j][o].  Each sum is one fmaf chain in order, its weights loaded
// 32 rows ahead (or from LDS): latency-bound, 256 pairs 26 -> 14 us with dZ.
__global__ void __launch_bounds__(256)
k_enc_head(const float* __restrict__ F, const float* __restrict__ W, const float* __restrict__ labels,
           const int* __restrict__ sel, int npairs, float* __restrict__ Z, float* __restrict__ OUT,
           float* __restrict__ DOUT, float* __restrict__ loss_part, float* __restrict__ DZ) {
  __shared__ float g[512];
  __shared__ float z[256];
  __shared__ float hw2[1536];
  __shared__ float dout[6];
  constexpr int kAhead = 32;
  const int b = blockIdx.x, t = threadIdx.x;
  const float* Hw1 = W + kEncHw1 + t;
  float next[kAhead];
#pragma unroll
  for (int u = 0; u < kAhead; ++u) next[u] = Hw1[u * 256];
  g[t] = F[(2 * b) * 256 + t];
  g[256 + t] = F[(2 * b + 1) * 256 + t];
#pragma unroll
  for (int u = 0; u < 6; ++u) hw2[u * 256 + t] = W[kEncHw2 + u * 256 + t];
  __syncthreads();
  float s = W[kEncHb1 + t];
  for (int i = 0; i < 512; i += kAhead) {
    float cur[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) cur[u] = next[u];
    const int n = min(i + kAhead, 512 - kAhead);  // past the end: the last rows again, unused
#pragma unroll
    for (int u = 0; u < kAhead; ++u) next[u] = Hw1[(n + u) * 256];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) s = fmaf(g[i + u], cur[u], s);
  }
  z[t] = relu(s);
  Z[b * 256 + t] = z[t];
  __syncthreads();
  if (t < 6) {
    float o = W[kEncHb2 + t];
#pragma unroll 16
    for (int i = 0; i < 256; ++i) o = fmaf(z[i], hw2[i * 6 + t], o);
    OUT[b * 6 + t] = o;
    if (labels) {
      const float d = o - labels[(int64_t)(sel ? sel[b] : b) * 6 + t];
      dout[t] = 2.f * d / (float)npairs;
      DOUT[b * 6 + t] = dout[t];
      loss_part[b * 6 + t] = d * d / (float)npairs;
    }
  }
  if (!labels) return;
  __syncthreads();
  float dz = 0.f;
#pragma unroll
  for (int o = 0; o < 6; ++o) dz = fmaf(dout[o], hw2[t * 6 + o], dz);
  DZ[b * 256 + t] = z[t] > 0.f ? dz : 0.f;
}

// dG[b][i] = sum_j dZ[b][j] Hw1[i][j] on FP32 matrix instructions: a block computes
// 16 pairs x 16 features, a wavefront 64 of the 256 terms (16-byte loads along
// them; component c of the four feeds instruction c on both sides), the four
// tiles added in wavefront order.
__global__ void __launch_bounds__(256)
k_enc_head_back(const float* __restrict__ DZ, const float* __restrict__ W, int npairs,
                float* __restrict__ DG) {
  __shared__ float red[4][256];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, l16 = lane & 15, q = lane >> 4;
  const int b = blockIdx.x * 16 + l16, i = blockIdx.y * 16 + l16;
  const float4* pa = reinterpret_cast<const float4*>(DZ + (int64_t)min(b, npairs - 1) * 256 + 64 * w + 4 * q);
  const float4* pb = reinterpret_cast<const float4*>(W + kEncHw1 + i * 256 + 64 * w + 4 * q);
  float4 a[4], v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    a[u] = pa[4 * u];
    v[u] = pb[4 * u];
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].x, v[u].x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].y, v[u].y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].z, v[u].z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].w, v[u].w, acc, 0, 0, 0);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) red[w][(4 * q + e) * 16 + l16] = acc[e];
  __syncthreads();
  const int ob = blockIdx.x * 16 + t / 16;
  if (ob < npairs)
    DG[(int64_t)ob * 512 + blockIdx.y * 16 + t % 16] = ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
}

// C[i][j] = sum_{r < R} A[r * lda + i] * B[r * ldb + j], and the column sums of B
// into bias[j] (a row of ones under A), on FP32 matrix instructions.  A block
// computes one 16 x 16 tile: each of its 4 wavefronts runs a quarter of the rows
// straight from memory (four rows per instruction, 64-byte row segments, eight
// steps of loads in flight), and their tiles are added in wavefront order.  The
// head's gradients at 256 pairs: 126 -> 9 us (one thread per output walked the
// rows one after the other).
__global__ void __launch_bounds__(256)
k_outer_mfma(const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb, int R, int M,
             int N, float* __restrict__ C, float* __restrict__ bias) {
  __shared__ float red[4][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, l16 = lane & 15, q = lane >> 4;
  const int i = blockIdx.x * 16 + l16, j = blockIdx.y * 16 + l16;
  const int per = ((R + 15) / 16) * 4;
  const int r0 = w * per, r1 = min(R, r0 + per);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  // every load at an address inside the arrays; what lies past M, N or the rows is
  // replaced afterwards
  const float* pa = A + min(i, M - 1);
  const float* pb = B + min(j, N - 1);
  for (int rb = r0; rb < r1; rb += 32) {
    float a[8], b[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int64_t rr = min(rb + 4 * u + q, R - 1);
      a[u] = pa[rr * lda];
      b[u] = pb[rr * ldb];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool ok = rb + 4 * u + q < r1;
      const float x = i < M ? a[u] : (i == M ? 1.f : 0.f);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ok ? x : 0.f, ok && j < N ? b[u] : 0.f, acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) red[w][(4 * q + e) * 16 + l16] = acc[e];
  __syncthreads();
  const int t = threadIdx.x, oi = blockIdx.x * 16 + t / 16, oj = blockIdx.y * 16 + t % 16;
  if (oi > M || oj >= N) return;
  const float s = ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
  if (oi < M)
    C[oi * N + oj] = s;
  else
    bias[oj] = s;
}

// Backward through the per-point layers.  The max-pool sends each channel's
// gradient to one point, so a cloud contributes 256 rows (channels).  A block
// takes 64 channels (blockIdx.x) of the clouds blockIdx.y, + gridDim.y, ... and
// keeps its share of every weight gradient in registers over all of them; only
// that share leaves the chip (part_w, part_w3, added in a fixed order by
// k_enc_grad_fold).  Per cloud:
//   layer 1 recomputed for the 64 argmax points (FP32), h1 as bf16 in LDS;
//   layer 2 on BF16 MFMA exactly as the forward computes it, transposed (columns
//   = rows of the batch), so a lane holds four consecutive channels of one point:
//   h2 df joins the W3 gradient, and m = (a2 > 0) W3 goes to LDS (bf16, exact);
//   dh1 = df (m W2^T): both factors are bf16, the products exact, df applied after
//   the FP32 sum; with h1's mask it joins the W1 gradient;
//   the W2 gradient h1^T (df m) on FP32 MFMA, operands widened from LDS.
// Bound by latency and the LDS and vector work around the MFMAs (about 6.5 GFLOP
// in all).  256 pairs (512 clouds): 1238 -> 57 us with the fold; before, the rows'
// activations and gradients (384 floats each) went through memory to four vector
// kernels.
constexpr int kGradW = kEncW3;                     // W1, b1, W2, b2: first in the flat layout
constexpr int kGradW3 = kEncB3 + 256 - kEncW3;     // W3, b3: next
constexpr int kGradGroups = 128;                   // cloud groups: 512 blocks, two per CU
constexpr int kGradMS = 128 + 8;                   // LDS row stride of m (bf16)

__global__ void __launch_bounds__(256, 2)
k_enc_grad(const float4* __restrict__ X, const int* __restrict__ sel, int npts,
           const float* __restrict__ F,
           const int* __restrict__ ARG, const float* __restrict__ DG, const float* __restrict__ W,
           const __bf16* __restrict__ W2t, const __bf16* __restrict__ W3t, int nclouds,
           float* __restrict__ part_w, float* __restrict__ part_w3) {
  __shared__ __attribute__((aligned(16))) __bf16 H1[64 * kH1S];
  __shared__ __attribute__((aligned(16))) __bf16 Mk[64 * kGradMS];
  __shared__ float4 xs[64];
  __shared__ float dfs[64];
  __shared__ float4 w1[64];  // (b1, W1) per output of layer 1: kept out of the registers
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, l16 = lane & 15, q = lane >> 4, kq = q * 8;
  const int c0 = blockIdx.x * 64;
  bf16x8 A2[2][2], B1[4];
  bf16x4 w3[4][2];
  f32x4 b2[2], acc3[4][2], accb2[2], acc2[4][2];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int jt = 0; jt < 2; ++jt) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      A2[jt][ks] = *(const bf16x8*)(W2t + (32 * w + 16 * jt + l16) * 64 + 32 * ks + kq);
    b2[jt] = *(const f32x4*)(W + kEncB2 + 32 * w + 16 * jt + 4 * q);
    accb2[jt] = zero;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      w3[rt][jt] = *(const bf16x4*)(W3t + (c0 + 16 * rt + l16) * 128 + 32 * w + 16 * jt + 4 * q);
      acc3[rt][jt] = zero;
      acc2[rt][jt] = zero;
    }
  }
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int v = 0; v < 8; ++v)
      B1[ks][v] = (__bf16)W[kEncW2 + (16 * w + l16) * 128 + 32 * ks + kq + v];
  float acc1[4] = {0.f, 0.f, 0.f, 0.f}, accb3 = 0.f;
  if (t < 64)
    w1[t] = make_float4(W[kEncB1 + t], W[kEncW1 + t], W[kEncW1 + 64 + t], W[kEncW1 + 128 + t]);
  for (int cloud = blockIdx.y; cloud < nclouds; cloud += gridDim.y) {
    if (t < 64) {
      const int c = cloud * 256 + c0 + t;
      const float df = F[c] > 0.f ? DG[c] : 0.f;
      xs[t] = cloud_points(X, sel, cloud, npts)[ARG[c]];
      dfs[t] = df;
      accb3 += df;
    }
    __syncthreads();
    {
      const int r = t >> 2, j0 = (t & 3) * 16;
      const float4 x = xs[r];
      bf16x8 h[2];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const float4 v = w1[j0 + u];
        float a = v.x;
        a = fmaf(x.x, v.y, a);
        a = fmaf(x.y, v.z, a);
        a = fmaf(x.z, v.w, a);
        h[u >> 3][u & 7] = (__bf16)relu(a);
      }
      *(bf16x8*)(H1 + r * kH1S + j0) = h[0];
      *(bf16x8*)(H1 + r * kH1S + j0 + 8) = h[1];
    }
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const int r = 16 * rt + l16;
      const float df = dfs[r];
      bf16x8 hf[2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) hf[ks] = *(const bf16x8*)(H1 + r * kH1S + 32 * ks + kq);
#pragma unroll
      for (int jt = 0; jt < 2; ++jt) {
        f32x4 acc = zero;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A2[jt][ks], hf[ks], acc, 0, 0, 0);
        bf16x4 m;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = acc[e] + b2[jt][e];
          const bool pos = a > 0.f;
          const float h2 = pos ? (float)(__bf16)a : 0.f;
          acc3[rt][jt][e] = fmaf(h2, df, acc3[rt][jt][e]);
          m[e] = pos ? w3[rt][jt][e] : (__bf16)0.f;
          accb2[jt][e] += df * (float)m[e];
        }
        *(bf16x4*)(Mk + r * kGradMS + 32 * w + 16 * jt + 4 * q) = m;
      }
      __builtin_amdgcn_sched_barrier(0);  // one row tile's operands live at a time
    }
    __syncthreads();
    // dh1 at columns i = 16 w + l16, and layer 1's gradient
#pragma unroll 1
    for (int rt = 0; rt < 4; ++rt) {
      f32x4 acc = zero;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 mf = *(const bf16x8*)(Mk + (16 * rt + l16) * kGradMS + 32 * ks + kq);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf, B1[ks], acc, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 16 * rt + 4 * q + e;
        const float4 x = xs[r];
        const float d = (float)H1[r * kH1S + 16 * w + l16] > 0.f ? acc[e] * dfs[r] : 0.f;
        acc1[0] = fmaf(x.x, d, acc1[0]);
        acc1[1] = fmaf(x.y, d, acc1[1]);
        acc1[2] = fmaf(x.z, d, acc1[2]);
        acc1[3] += d;
      }
    }
    // W2 gradient: columns j = 32 w + 16 jt + l16, rows of the batch four at a time
#pragma unroll 2
    for (int ks = 0; ks < 16; ++ks) {
      const int r = 4 * ks + q;
      const float df = dfs[r];
      float bv[2];
#pragma unroll
      for (int jt = 0; jt < 2; ++jt) bv[jt] = df * (float)Mk[r * kGradMS + 32 * w + 16 * jt + l16];
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const float av = (float)H1[r * kH1S + 16 * it + l16];
#pragma unroll
        for (int jt = 0; jt < 2; ++jt)
          acc2[it][jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv[jt], acc2[it][jt], 0, 0, 0);
      }
    }
    __syncthreads();  // xs, dfs, H1 and Mk are rewritten for the next cloud
  }
  float* pw = part_w + (int64_t)(blockIdx.y * gridDim.x + blockIdx.x) * kGradW;
  float* p3 = part_w3 + (int64_t)blockIdx.y * kGradW3;
#pragma unroll
  for (int it = 0; it < 4; ++it)
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pw[kEncW2 + (16 * it + 4 * q + e) * 128 + 32 * w + 16 * jt + l16] = acc2[it][jt][e];
        p3[(32 * w + 16 * jt + 4 * q + e) * 256 + c0 + 16 * it + l16] = acc3[it][jt][e];
      }
#pragma unroll
  for (int jt = 0; jt < 2; ++jt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = accb2[jt][e];
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
      if (l16 == 0) pw[kEncB2 + 32 * w + 16 * jt + 4 * q + e] = v;
    }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    float v = acc1[c];
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (q == 0) pw[kEncW1 + c * 64 + 16 * w + l16] = v;  // W1's three rows, then b1
  }
  if (t < 64) p3[kEncB3 - kEncW3 + c0 + t] = accb3;
}

// The blocks' shares added in a fixed order: 64 outputs per block, eight slices of
// the shares each.  part_w has 4 * groups shares, part_w3 one per group.
constexpr int kFoldSlices = 8;

__global__ void __launch_bounds__(64 * kFoldSlices)
k_enc_grad_fold(const float* __restrict__ part_w, const float* __restrict__ part_w3, int groups,
                float* __restrict__ G) {
  static_assert(kGradW % 64 == 0 && kGradW3 % 64 == 0, "a block's outputs lie in one part");
  __shared__ float red[kFoldSlices][64];
  const int o = blockIdx.x * 64 + (threadIdx.x & 63), slice = threadIdx.x >> 6;
  const bool w3 = o >= kGradW;
  const int n = w3 ? groups : 4 * groups, stride = w3 ? kGradW3 : kGradW;
  const float* p = w3 ? part_w3 + (o - kGradW) : part_w + o;
  float s = 0.f;
#pragma unroll 8
  for (int k = slice; k < n; k += kFoldSlices) s += p[(int64_t)k * stride];
  red[slice][threadIdx.x & 63] = s;
  __syncthreads();
  if (slice != 0) return;
#pragma unroll
  for (int k = 1; k < kFoldSlices; ++k) s += red[k][threadIdx.x];
  G[o] = s;
}

// Adam (FP32 master weights, and the BF16 transposed copies of W2 and W3 with them);
// the block past the parameters sums the step's loss terms in a fixed order.
__global__ void __launch_bounds__(256)
k_adam(float* __restrict__ W, const float* __restrict__ G, float* __restrict__ M,
       float* __restrict__ V, int n, float lr, float b1, float b2, float eps, float c1, float c2,
       __bf16* __restrict__ W2t, __bf16* __restrict__ W3t, const float* __restrict__ loss_part,
       int nloss, float* __restrict__ loss) {
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ float s[256];
    float a = 0.f;
    for (int i = threadIdx.x; i < nloss; i += 256) a += loss_part[i];
    s[threadIdx.x] = a;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = s[0];
    return;
  }
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = G[i];
  const float m = b1 * M[i] + (1.f - b1) * g;
  const float v = b2 * V[i] + (1.f - b2) * g * g;
  M[i] = m;
  V[i] = v;
  const float x = W[i] - lr * (m / c1) / (sqrtf(v / c2) + eps);
  W[i] = x;
  if (i >= kEncW2 && i < kEncB2) {
    const int k = i - kEncW2;  // W2[i][j] -> W2t[j][i]
    W2t[(k & 127) * 64 + (k >> 7)] = (__bf16)x;
  } else if (i >= kEncW3 && i < kEncB3) {
    const int k = i - kEncW3;  // W3[k][c] -> W3t[c][k]
    W3t[(k & 255) * 128 + (k >> 8)] = (__bf16)x;
  }
}

__global__ void k_enc_bf16_weights(const float* __restrict__ W, __bf16* __restrict__ W2t,
                                   __bf16* __restrict__ W3t) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < 64 * 128) {
    const int i = idx / 128, j = idx % 128;  // W2[i][j] -> W2t[j][i]
    W2t[j * 64 + i] = (__bf16)W[kEncW2 + idx];
  }
  if (idx < 128 * 256) {
    const int k = idx / 256, c = idx % 256;  // W3[k][c] -> W3t[c][k]
    W3t[c * 128 + k] = (__bf16)W[kEncW3 + idx];
  }
}

// Cloud groups of the per-point backward: one per cloud up to kGradGroups.
inline int enc_grad_groups(int nclouds) { return nclouds < kGradGroups ? nclouds : kGradGroups; }

inline unsigned nb(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

}  // namespace

int enc_forward_chunks(int npts) { return (npts + kRows - 1) / kRows; }

void launch_enc_bf16_weights(const float* W, __bf16* W2t, __bf16* W3t, hipStream_t s) {
  hipLaunchKernelGGL(k_enc_bf16_weights, dim3(nb(128 * 256, 256)), dim3(256), 0, s, W, W2t, W3t);
}

void launch_enc_forward(const EncBuffers& e, int npairs, int npts, const float* labels,
                        hipStream_t s) {
  const int nclouds = 2 * npairs;
  // Passes per block: up to kMaxPasses, as long as the blocks still fill the chip
  // four times over at three per CU (more passes load the weights less often and
  // leave fewer partials to fold; fewer blocks leave an emptier last round).
  const int64_t units = (int64_t)enc_forward_chunks(npts) * nclouds;
  const int iters = (int)std::min<int64_t>(std::max<int64_t>(units / (256 * 3 * 4), 1), kMaxPasses);
  const int nchunks = (enc_forward_chunks(npts) + iters - 1) / iters;
  hipLaunchKernelGGL(k_enc_points, dim3(nchunks, nclouds), dim3(256), 0, s, e.X, e.sel, npts, iters,
                     e.W, e.W2t, e.W3t, e.part_max, e.part_arg);
  hipLaunchKernelGGL(k_enc_pool, dim3(nclouds), dim3(256), 0, s, e.part_max, e.part_arg, nchunks,
                     e.F, e.ARG);
  hipLaunchKernelGGL(k_enc_head, dim3(npairs), dim3(256), 0, s, e.F, e.W, labels, e.sel, npairs,
                     e.Z, e.OUT, e.DOUT, e.loss_part, e.DZ);
}

void launch_enc_backward(const EncBuffers& e, int npairs, int npts, hipStream_t s) {
  const int nclouds = 2 * npairs;
  float* G = e.G;
  hipLaunchKernelGGL(k_enc_head_back, dim3(nb(npairs, 16), 32), dim3(256), 0, s, e.DZ, e.W, npairs, e.DG);
  // head weights: dHw2 = Z^T dOut, dHw1 = G^T dZ (G = pooled features)
  hipLaunchKernelGGL(k_outer_mfma, dim3(17, 1), dim3(256), 0, s, e.Z, 256, e.DOUT, 6, npairs, 256, 6,
                     G + kEncHw2, G + kEncHb2);
  hipLaunchKernelGGL(k_outer_mfma, dim3(33, 16), dim3(256), 0, s, e.F, 512, e.DZ, 256, npairs, 512,
                     256, G + kEncHw1, G + kEncHb1);
  // per-point layers
  const int groups = enc_grad_groups(nclouds);
  float* part_w3 = e.part_grad + (int64_t)4 * groups * kGradW;
  hipLaunchKernelGGL(k_enc_grad, dim3(4, groups), dim3(256), 0, s, e.X, e.sel, npts, e.F, e.ARG, e.DG,
                     e.W, e.W2t, e.W3t, nclouds, e.part_grad, part_w3);
  hipLaunchKernelGGL(k_enc_grad_fold, dim3((kGradW + kGradW3) / 64), dim3(64 * kFoldSlices), 0, s,
                     e.part_grad, part_w3, groups, G);
}

void launch_adam(const EncBuffers& e, float* M, float* V, int npairs, float lr, int step, float* loss,
                 hipStream_t s) {
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(nb(kEncNParam, 256) + 1), dim3(256), 0, s, e.W, e.G, M, V, kEncNParam,
                     lr, b1, b2, eps, c1, c2, e.W2t, e.W3t, e.loss_part, npairs * 6, loss);
}

int64_t enc_part_grad_floats(int npairs) {
  return (int64_t)enc_grad_groups(2 * npairs) * (4 * kGradW + kGradW3);
}

}  // namespace lcr
