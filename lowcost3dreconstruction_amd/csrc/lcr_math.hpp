// lcr_math.hpp -- FP64 small-matrix solvers used at the end of every ICP
// iteration, and the convergence state machine.  All loops have compile-time
// trip counts and are unrolled, so every array index is a constant and the
// matrices stay in registers (no private scratch memory).
//
// Solvers:
//   * horn_rotation   -- point-to-point: the rotation maximising trace(R^T S) from
//     the 3x3 cross-covariance S, as the eigenvector of Horn's 4x4 matrix with the
//     largest eigenvalue (Horn 1987): Newton on the characteristic polynomial and
//     the adjugate where that eigenvalue is well separated, cyclic Jacobi
//     otherwise.  Equals Umeyama's U diag(1,1,det) V^T, which
//     TransformationEstimationSVD computes (pcl/registration/impl/
//     transformation_estimation_svd.hpp; called via fine_registration.cpp:121).
//   * chol6_solve     -- point-to-plane: the 6x6 normal equations of
//     TransformationEstimationPointToPlaneLLS, by Cholesky.
//   * smallest_eigvec3, eigh3 -- normals: the smallest eigenvalue's eigenvector of
//     the covariance from its characteristic polynomial where that eigenvalue is
//     well separated, cyclic Jacobi otherwise (NormalEstimation's solvePlaneParameters, normal_estimation.cpp:108).
//   * conv_step       -- DefaultConvergenceCriteria::hasConverged.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "lcr_common.hpp"

namespace lcr {

#define LCR_HD __host__ __device__ inline

// Cyclic Jacobi on a symmetric 4x4 (upper and lower kept in sync).  On exit a is
// diagonal (eigenvalues) and v's columns are the eigenvectors.
LCR_HD void jacobi4(double a[4][4], double v[4][4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[i][j] = (i == j) ? 1.0 : 0.0;
  for (int sweep = 0; sweep < 24; ++sweep) {
    double off = 0.0, dg = 0.0;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      dg += a[p][p] * a[p][p];
#pragma unroll
      for (int q = p + 1; q < 4; ++q) off += a[p][q] * a[p][q];
    }
    if (off == 0.0 || off <= 1e-32 * dg) break;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int q = p + 1; q < 4; ++q) {
        const double apq = a[p][q];
        if (apq != 0.0) {
          const double theta = (a[q][q] - a[p][p]) / (2.0 * apq);
          const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
          const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const double akp = a[k][p], akq = a[k][q];
            a[k][p] = c * akp - s * akq;
            a[k][q] = s * akp + c * akq;
          }
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const double apk = a[p][k], aqk = a[q][k];
            a[p][k] = c * apk - s * aqk;
            a[q][k] = s * apk + c * aqk;
          }
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const double vkp = v[k][p], vkq = v[k][q];
            v[k][p] = c * vkp - s * vkq;
            v[k][q] = s * vkp + c * vkq;
          }
        }
      }
    }
  }
}

// The eigenvector of the largest eigenvalue of a symmetric traceless 4x4 matrix a
// with entries of at most 1 in magnitude.  The eigenvalue is the largest root of
// l^4 + c2 l^2 + c1 l + c0 (all roots real): Newton from a bound above it descends
// monotonically.  The adjugate of a - l I is the eigenvector's outer product times
// the product of the eigenvalue's distances to the others, p'(l); its column of
// largest diagonal is taken, and one step against its residual follows: the
// column's rounding is relative to p'(l), after the step it is relative to the
// nearest distance alone, as Jacobi's is (against 64-bit mantissas, singular values
// (1, .04, .01): 6.4e-15 without the step, 1.1e-15 with it, Jacobi 2.0e-15; (1, 1,
// -.9): 9.6e-14, 9.8e-16, 1.6e-15; (1, .6, .3): 2.2e-16, 2.0e-16, 3.2e-16).  Where
// p'(l) is below kSeparated (degenerate clouds) this returns false and the caller
// takes Jacobi.  About 0.7 us of one lane's FP64 latency against 9 for Jacobi's
// 25-30 rotations of two divisions and two square roots.
constexpr double kSeparated = 0.05;

LCR_HD bool top_eigvec4(const double a[4][4], double q[4]) {
  double fro = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) fro += a[i][j] * a[i][j];
  // power sums of the eigenvalues: p2 = fro, p3 = trace(a^3)
  double p3 = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < 4; ++k) s += a[i][k] * a[k][j];
      p3 += s * a[j][i];
    }
  // 2x2 minors of the first and the last two rows: determinant and adjugate
  auto det = [](const double m[4][4]) {
    const double s0 = m[0][0] * m[1][1] - m[1][0] * m[0][1], s1 = m[0][0] * m[1][2] - m[1][0] * m[0][2];
    const double s2 = m[0][0] * m[1][3] - m[1][0] * m[0][3], s3 = m[0][1] * m[1][2] - m[1][1] * m[0][2];
    const double s4 = m[0][1] * m[1][3] - m[1][1] * m[0][3], s5 = m[0][2] * m[1][3] - m[1][2] * m[0][3];
    const double c5 = m[2][2] * m[3][3] - m[3][2] * m[2][3], c4 = m[2][1] * m[3][3] - m[3][1] * m[2][3];
    const double c3 = m[2][1] * m[3][2] - m[3][1] * m[2][2], c2 = m[2][0] * m[3][3] - m[3][0] * m[2][3];
    const double c1 = m[2][0] * m[3][2] - m[3][0] * m[2][2], c0 = m[2][0] * m[3][1] - m[3][0] * m[2][1];
    return s0 * c5 - s1 * c4 + s2 * c3 + s3 * c2 - s4 * c1 + s5 * c0;
  };
  const double c2 = -0.5 * fro, c1 = -p3 / 3.0, c0 = det(a);
  // a traceless matrix's largest eigenvalue is at most sqrt(3 / 4) of its norm
  double l = 0.8660254037844387 * sqrt(fro) * (1.0 + 1e-12);
  double dp = 0.0;
  for (int it = 0; it < 40; ++it) {
    const double l2 = l * l;
    const double f = (l2 + c2) * l2 + (c1 * l + c0);
    dp = (4.0 * l2 + 2.0 * c2) * l + c1;
    if (!(dp > 0.0)) return false;
    const double step = f / dp;
    l -= step;
    if (!(fabs(step) > 4e-16 * l)) break;
  }
  if (!(dp > kSeparated)) return false;
  double m[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) m[i][j] = a[i][j] - (i == j ? l : 0.0);
  // cofactor of (i, j): symmetric, so the adjugate's column j
  auto cof = [&](int i, int j) {
    const int r0 = i == 0 ? 1 : 0, r1 = i <= 1 ? 2 : 1, r2 = i <= 2 ? 3 : 2;
    const int k0 = j == 0 ? 1 : 0, k1 = j <= 1 ? 2 : 1, k2 = j <= 2 ? 3 : 2;
    const double d = m[r0][k0] * (m[r1][k1] * m[r2][k2] - m[r1][k2] * m[r2][k1]) -
                     m[r0][k1] * (m[r1][k0] * m[r2][k2] - m[r1][k2] * m[r2][k0]) +
                     m[r0][k2] * (m[r1][k0] * m[r2][k1] - m[r1][k1] * m[r2][k0]);
    return ((i + j) & 1) ? -d : d;
  };
  double c[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = i; j < 4; ++j) c[i][j] = c[j][i] = cof(i, j);
  double best = 0.0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (fabs(c[j][j]) > best) {
      best = fabs(c[j][j]);
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = c[i][j];
    }
  }
  // one step against the residual r = m q: the inverse of m across q from its
  // characteristic polynomial, (m^2 + 4 l m + 6 l^2 + c2) / -p'(l)
  auto times = [&](const double v[4], double out[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[i] = (m[i][0] * v[0] + m[i][1] * v[1]) + (m[i][2] * v[2] + m[i][3] * v[3]);
  };
  double r[4], mr[4], mmr[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r[i] = (a[i][0] * q[0] + a[i][1] * q[1]) + (a[i][2] * q[2] + a[i][3] * q[3]) - l * q[i];
  times(r, mr);
  times(mr, mmr);
  const double e2 = 6.0 * l * l + c2, inv = 1.0 / dp;
#pragma unroll
  for (int i = 0; i < 4; ++i) q[i] += (mmr[i] + 4.0 * l * mr[i] + e2 * r[i]) * inv;
  return best > 0.0;
}

// S[a][b] = cross-covariance sum_i (s_i - mu_s)_a (t_i - mu_t)_b / n, source first.
// Returns the row-major rotation R (3x3) taking the source onto the target.
LCR_HD void horn_rotation(const double S[3][3], double R[3][3]) {
  const double sxx = S[0][0], sxy = S[0][1], sxz = S[0][2];
  const double syx = S[1][0], syy = S[1][1], syz = S[1][2];
  const double szx = S[2][0], szy = S[2][1], szz = S[2][2];
  double N[4][4] = {
      {sxx + syy + szz, syz - szy, szx - sxz, sxy - syx},
      {syz - szy, sxx - syy - szz, sxy + syx, szx + sxz},
      {szx - sxz, sxy + syx, -sxx + syy - szz, syz + szy},
      {sxy - syx, szx + sxz, syz + szy, -sxx - syy + szz}};
  // scale for a well-conditioned Jacobi (the eigenvectors are scale-free)
  double m = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) m = fmax(m, fabs(N[i][j]));
  const double inv = m > 0.0 ? 1.0 / m : 1.0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) N[i][j] *= inv;
  double q[4];
  if (!top_eigvec4(N, q)) {
    double V[4][4];
    jacobi4(N, V);
    double best = N[0][0];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = V[i][0];
#pragma unroll
    for (int c = 1; c < 4; ++c) {
      if (N[c][c] > best) {
        best = N[c][c];
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = V[i][c];
      }
    }
  }
  double q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
  const double nq = sqrt(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3);
  q0 /= nq;
  q1 /= nq;
  q2 /= nq;
  q3 /= nq;
  R[0][0] = q0 * q0 + q1 * q1 - q2 * q2 - q3 * q3;
  R[0][1] = 2.0 * (q1 * q2 - q0 * q3);
  R[0][2] = 2.0 * (q1 * q3 + q0 * q2);
  R[1][0] = 2.0 * (q2 * q1 + q0 * q3);
  R[1][1] = q0 * q0 - q1 * q1 + q2 * q2 - q3 * q3;
  R[1][2] = 2.0 * (q2 * q3 - q0 * q1);
  R[2][0] = 2.0 * (q3 * q1 - q0 * q2);
  R[2][1] = 2.0 * (q3 * q2 + q0 * q1);
  R[2][2] = q0 * q0 - q1 * q1 - q2 * q2 + q3 * q3;
}

// Point-to-point increment from the FP64 raw moments of one iteration:
// v[0] n, v[1..3] sum s, v[4..6] sum t, v[7..15] sum s_a t_b, as laid out in
// lcr_common.hpp.  T is row-major 4x4.
LCR_HD void p2p_increment(const double* v, double T[16]) {
  const double n = v[0];
  const double ms[3] = {v[1] / n, v[2] / n, v[3] / n};
  const double mt[3] = {v[4] / n, v[5] / n, v[6] / n};
  double S[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) S[a][b] = v[7 + 3 * a + b] / n - ms[a] * mt[b];
  double R[3][3];
  horn_rotation(S, R);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < 3; ++j) T[4 * i + j] = R[i][j];
    T[4 * i + 3] = mt[i] - (R[i][0] * ms[0] + R[i][1] * ms[1] + R[i][2] * ms[2]);
  }
  T[12] = 0.0;
  T[13] = 0.0;
  T[14] = 0.0;
  T[15] = 1.0;
}

// upper-triangle index of (i, j), i <= j, in a 6x6 row-major packing
LCR_HD constexpr int tri6(int i, int j) { return i * 6 - (i * (i - 1)) / 2 + (j - i); }

// Solve M x = b for symmetric positive definite M given as its packed upper
// triangle.  Returns false when a pivot is not positive.  One division per pivot
// (the reciprocal of its root scales the column and both substitutions): divisions
// and roots are what one lane's latency goes to.
LCR_HD bool chol6_solve(const double* up, const double* b, double x[6]) {
  double L[6][6], inv[6];
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int j = 0; j < 6; ++j) L[i][j] = 0.0;
  bool ok = true;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    double d = up[tri6(j, j)];
#pragma unroll
    for (int k = 0; k < j; ++k) d -= L[j][k] * L[j][k];
    if (!(d > 0.0)) ok = false;
    inv[j] = 1.0 / sqrt(d > 0.0 ? d : 1.0);
#pragma unroll
    for (int i = j + 1; i < 6; ++i) {
      double s = up[tri6(j, i)];
#pragma unroll
      for (int k = 0; k < j; ++k) s -= L[i][k] * L[j][k];
      L[i][j] = s * inv[j];
    }
  }
  double y[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    double s = b[i];
#pragma unroll
    for (int k = 0; k < i; ++k) s -= L[i][k] * y[k];
    y[i] = s * inv[i];
  }
#pragma unroll
  for (int i = 5; i >= 0; --i) {
    double s = y[i];
#pragma unroll
    for (int k = i + 1; k < 6; ++k) s -= L[k][i] * x[k];
    x[i] = s * inv[i];
  }
  return ok;
}

// TransformationEstimationPointToPlaneLLS::constructTransformationMatrix:
// T = [Rz(g) Ry(b) Rx(a) | t].
LCR_HD void p2pl_matrix(const double sn[3], const double cs[3], const double x[6], double T[16]) {
  const double ca = cs[0], sa = sn[0];
  const double cb = cs[1], sb = sn[1];
  const double cg = cs[2], sg = sn[2];
  T[0] = cg * cb;
  T[1] = -sg * ca + cg * sb * sa;
  T[2] = sg * sa + cg * sb * ca;
  T[3] = x[3];
  T[4] = sg * cb;
  T[5] = cg * ca + sg * sb * sa;
  T[6] = -cg * sa + sg * sb * ca;
  T[7] = x[4];
  T[8] = -sb;
  T[9] = cb * sa;
  T[10] = cb * ca;
  T[11] = x[5];
  T[12] = 0.0;
  T[13] = 0.0;
  T[14] = 0.0;
  T[15] = 1.0;
}

// Point-to-plane increment from v[1..21] (packed A^T A) and v[22..27] (A^T b).
// Returns false if the system is not positive definite (T = identity then).  On
// the device every lane of a wavefront calls it with the same v: lane l takes the
// sine and cosine of angle l % 3, so the three angles cost one's latency.
LCR_HD bool p2pl_increment(const double* v, double T[16]) {
  double x[6];
  const bool ok = chol6_solve(v + 1, v + 22, x);
  if (!ok) {
#pragma unroll
    for (int i = 0; i < 16; ++i) T[i] = (i % 5 == 0) ? 1.0 : 0.0;
    return false;
  }
  double sn[3], cs[3];
#ifdef __HIP_DEVICE_COMPILE__
  const int l = (int)(threadIdx.x & 63) % 3;
  double s1, c1;
  sincos(l == 0 ? x[0] : (l == 1 ? x[1] : x[2]), &s1, &c1);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    sn[i] = __shfl(s1, i, 64);
    cs[i] = __shfl(c1, i, 64);
  }
#else
  for (int i = 0; i < 3; ++i) {
    sn[i] = sin(x[i]);
    cs[i] = cos(x[i]);
  }
#endif
  p2pl_matrix(sn, cs, x, T);
  return true;
}

LCR_HD void mat4_mul(const double* A, const double* B, double* C) {
  double t[16];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      double s = 0.0;
#pragma unroll
      for (int k = 0; k < 4; ++k) s += A[4 * i + k] * B[4 * k + j];
      t[4 * i + j] = s;
    }
#pragma unroll
  for (int i = 0; i < 16; ++i) C[i] = t[i];
}

// Smallest eigenvalue w and its unit eigenvector v of a symmetric positive
// semi-definite 3x3 matrix.  With entries scaled to at most 1 and the mean
// eigenvalue taken off, the smallest root of the characteristic polynomial
// x^3 - (p2 / 2) x - det by Newton from a bound below it (f is increasing and
// concave there, so the steps never pass it); the adjugate at that root is
// v v^T times the product of its distances to the other two, f'(x), and w is v's
// Rayleigh quotient.  v's rounding is relative to f'(x); after one step against its
// residual it is relative to the nearer distance alone, as Jacobi's is (eigenvalues
// (0, .05, 1): 2.8e-15 without the step, 2.2e-16 with it, Jacobi 2.4e-16; (0, .5, 1):
// 1.1e-16, 0.8e-16, 2.1e-16).  Below kSeparated3 (points on a line, or one cloud of
// them) this returns false and the caller takes Jacobi.  Three divisions and two
// square roots plus 4-6 divisions of Newton, against about nine rotations of two
// divisions and two square roots each.
constexpr double kSeparated3 = 0.01;

LCR_HD bool smallest_eigvec3(const double C[3][3], double& w, double v[3]) {
  const double m = fmax(fmax(C[0][0], C[1][1]), C[2][2]);
  if (!(m > 0.0)) return false;
  const double inv = 1.0 / m;
  const double q = (C[0][0] + C[1][1] + C[2][2]) * inv * (1.0 / 3.0);
  const double d0 = C[0][0] * inv - q, d1 = C[1][1] * inv - q, d2 = C[2][2] * inv - q;
  const double a01 = C[0][1] * inv, a02 = C[0][2] * inv, a12 = C[1][2] * inv;
  const double h = 0.5 * (d0 * d0 + d1 * d1 + d2 * d2) + (a01 * a01 + a02 * a02 + a12 * a12);
  const double det = d0 * (d1 * d2 - a12 * a12) - a01 * (a01 * d2 - a12 * a02) +
                     a02 * (a01 * a12 - d1 * a02);
  // the roots lie within 2 sqrt(h / 3) of 0
  double x = -1.1547005383792517 * sqrt(h) * (1.0 + 1e-12);
  double dp = 0.0;
  for (int it = 0; it < 40; ++it) {
    const double x2 = x * x;
    dp = 3.0 * x2 - h;
    if (!(dp > kSeparated3)) return false;
    const double step = ((x2 - h) * x - det) / dp;
    x -= step;
    if (!(fabs(step) > 4e-16)) break;
  }
  const double b0 = d0 - x, b1 = d1 - x, b2 = d2 - x;
  const double c00 = b1 * b2 - a12 * a12, c11 = b0 * b2 - a02 * a02, c22 = b0 * b1 - a01 * a01;
  const double c01 = a02 * a12 - a01 * b2, c02 = a01 * a12 - a02 * b1, c12 = a01 * a02 - a12 * b0;
  double v0 = c00, v1 = c01, v2 = c02, best = c00;
  if (c11 > best) {
    best = c11;
    v0 = c01;
    v1 = c11;
    v2 = c12;
  }
  if (c22 > best) {
    v0 = c02;
    v1 = c12;
    v2 = c22;
  }
  const double n = 1.0 / sqrt(v0 * v0 + v1 * v1 + v2 * v2);
  v[0] = v0 * n;
  v[1] = v1 * n;
  v[2] = v2 * n;
  w = v[0] * (C[0][0] * v[0] + C[0][1] * v[1] + C[0][2] * v[2]) +
      v[1] * (C[0][1] * v[0] + C[1][1] * v[1] + C[1][2] * v[2]) +
      v[2] * (C[0][2] * v[0] + C[1][2] * v[1] + C[2][2] * v[2]);
  // one step against the residual r of E v, E = C less the root (its entries rounded
  // once): across v the inverse of E is (trace(E) - E) / (m^2 f'(x))
  const double mu = (q + x) * m;
  const double e0 = C[0][0] - mu, e1 = C[1][1] - mu, e2 = C[2][2] - mu;
  double r0 = e0 * v[0] + C[0][1] * v[1] + C[0][2] * v[2];
  double r1 = C[0][1] * v[0] + e1 * v[1] + C[1][2] * v[2];
  double r2 = C[0][2] * v[0] + C[1][2] * v[1] + e2 * v[2];
  const double along = r0 * v[0] + r1 * v[1] + r2 * v[2];
  r0 -= along * v[0];
  r1 -= along * v[1];
  r2 -= along * v[2];
  const double s = e0 + e1 + e2, p = inv * inv / dp;
  v[0] -= (s * r0 - (e0 * r0 + C[0][1] * r1 + C[0][2] * r2)) * p;
  v[1] -= (s * r1 - (C[0][1] * r0 + e1 * r1 + C[1][2] * r2)) * p;
  v[2] -= (s * r2 - (C[0][2] * r0 + C[1][2] * r1 + e2 * r2)) * p;
  return true;
}

// Symmetric 3x3 eigen-decomposition (cyclic Jacobi, FP64).  a is row-major and
// overwritten; returns eigenvalues ascending in w and eigenvectors as columns of v.
LCR_HD void eigh3(double a[3][3], double w[3], double v[3][3]) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) v[i][j] = (i == j) ? 1.0 : 0.0;
  for (int sweep = 0; sweep < 24; ++sweep) {
    const double off = a[0][1] * a[0][1] + a[0][2] * a[0][2] + a[1][2] * a[1][2];
    const double dg = a[0][0] * a[0][0] + a[1][1] * a[1][1] + a[2][2] * a[2][2];
    if (off == 0.0 || off <= 1e-34 * dg) break;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int q = p + 1; q < 3; ++q) {
        const double apq = a[p][q];
        if (apq != 0.0) {
          const double theta = (a[q][q] - a[p][p]) / (2.0 * apq);
          const double t = (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
          const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const double akp = a[k][p], akq = a[k][q];
            a[k][p] = c * akp - s * akq;
            a[k][q] = s * akp + c * akq;
          }
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const double apk = a[p][k], aqk = a[q][k];
            a[p][k] = c * apk - s * aqk;
            a[q][k] = s * apk + c * aqk;
          }
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const double vkp = v[k][p], vkq = v[k][q];
            v[k][p] = c * vkp - s * vkq;
            v[k][q] = s * vkp + c * vkq;
          }
        }
      }
    }
  }
  w[0] = a[0][0];
  w[1] = a[1][1];
  w[2] = a[2][2];
  // sort ascending, permuting eigenvector columns: compare-swaps (0,1) (1,2) (0,1)
#pragma unroll
  for (int pass = 0; pass < 3; ++pass) {
    const int i = (pass == 1) ? 1 : 0;
    const int j = (pass == 1) ? 2 : 1;
    if (w[j] < w[i]) {
      const double tw = w[i];
      w[i] = w[j];
      w[j] = tw;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double tv = v[k][i];
        v[k][i] = v[k][j];
        v[k][j] = tv;
      }
    }
  }
}

// DefaultConvergenceCriteria::hasConverged (default_convergence_criteria.hpp) with
// max_iterations_similar_transforms_ = 0 and failure_after_max_iter_ = false.  The
// rotation and translation tests read the increment's coefficients as float, as
// PCL's Matrix4f does.  Returns true when converged; st->state says why.
LCR_HD bool conv_step(PairState* st, const IcpConst& c, const double* Tinc, double mse) {
  bool similar = false;
  if (st->iterations >= c.max_iterations) {
    st->state = kIterations;
    return true;
  }
  const float t00 = (float)Tinc[0], t11 = (float)Tinc[5], t22 = (float)Tinc[10];
  const float t03 = (float)Tinc[3], t13 = (float)Tinc[7], t23 = (float)Tinc[11];
  const float tr = ((t00 + t11) + t22) - 1.0f;
  const double cos_angle = 0.5 * (double)tr;
  const float tsq = (t03 * t03 + t13 * t13) + t23 * t23;
  const double translation_sqr = (double)tsq;
  if (cos_angle >= c.rotation_threshold && translation_sqr <= c.translation_threshold) {
    if (st->similar >= 0) {
      st->state = kTransform;
      return true;
    }
    similar = true;
  }
  const double dm = fabs(mse - st->prev_mse);
  if (dm < c.mse_abs) {
    if (st->similar >= 0) {
      st->state = kAbsMse;
      return true;
    }
    similar = true;
  }
  if (dm / st->prev_mse < c.mse_rel) {
    if (st->similar >= 0) {
      st->state = kRelMse;
      return true;
    }
    similar = true;
  }
  st->similar = similar ? st->similar + 1 : 0;
  st->prev_mse = mse;
  return false;
}

}  // namespace lcr
