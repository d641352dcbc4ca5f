// SE(3) helpers of the CLIK kernels (device; the batched kernels' log in FP32):
// body-frame images of motion vectors, the SE(3) log and its Jacobian, and the
// damped 6x6 solve, as used by compute_inverse_kinematics
// (pinocchio_model.cpp:228-300).
#pragma once
#include <hip/hip_runtime.h>

#include "spatial.h"

namespace sapamd {

// Body (local) frame image of a world motion vector under link pose (R, p):
// Ad(M)^-1 m = [R^T (l - p x a); R^T a].
template <class T> __device__ __forceinline__ S6<T> to_local(const T *R, V3<T> p, S6<T> m) {
  return {mtv(R, m.l - cross(p, m.a)), mtv(R, m.a)};
}

template <class T> __device__ __forceinline__ void vec_of(S6<T> x, T *v) {
  v[0] = x.l.x; v[1] = x.l.y; v[2] = x.l.z; v[3] = x.a.x; v[4] = x.a.y; v[5] = x.a.z;
}

// ---------------------------------------------------------------- SE(3) log for CLIK
// The FP32 quotients of the log without the general division's scaling and
// fix-up (3 to 6 instructions instead of about 10): the hardware reciprocal and
// one residual correction each. Over every angle of [0, pi] the coefficients
// below come out as IEEE division gives them, bit for bit (all 2^30 floats
// compared), so a CLIK problem takes the same iterations.
__device__ __forceinline__ float rn_rcp(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}
__device__ __forceinline__ float rn_div(float a, float b) {
  const float r = rn_rcp(b), q = a * r;
  return fmaf(fmaf(-b, q, a), r, q);
}
__device__ __forceinline__ float rn_div_by(float a, float b) {  // b a constant
  const float r = 1.f / b, q = a * r;
  return fmaf(fmaf(-q, b, a), r, q);
}
__device__ __forceinline__ double rn_div_by(double a, double b) { return a / b; }

// Rotation log in the form Pinocchio 2.6 evaluates it (the reference's
// log6 / Jlog6 inside compute_inverse_kinematics): theta = acos((tr R - 1) / 2)
// clipped to [0, pi]; below pi - 1e-2 the axial vector
// theta / (2 sin theta) (R - R^T)^v, with the factor 1 below theta = 2^-13
// (eps^(1/4)) in FP64 and 1 + theta^2 / 6 below 1e-3 in FP32; above, the axis
// magnitudes from the diagonal, R_ii = cos theta + (1 - cos theta) k_i^2, with
// the signs of the skew part. For a rotation any correct log agrees; this
// form also gives the reference's error vector when R is not orthonormal (a
// target built from a quaternion that is not unit length).
// s, c: sin and cos of the angle, for the coefficients as well. FP32; the
// per-call kernel has its own FP64 form.
__device__ __forceinline__ V3<float> log3_dev(const float *R, float &theta, float &s, float &c) {
  const float PI = 3.14159265358979323846f;
  const float tr = R[0] + R[4] + R[8];
  theta = tr >= 3.f ? 0.f : tr <= -1.f ? PI : acos((tr - 1.f) * 0.5f);
  sincosf(theta, &s, &c);
  const V3<float> ax = {0.5f * (R[7] - R[5]), 0.5f * (R[2] - R[6]), 0.5f * (R[3] - R[1])};
  if (theta < PI - 1e-2f) {
    const float k = theta > 1e-3f ? rn_div(theta, s) : 1.f + theta * theta / 6.f;
    return k * ax;
  }
  const float b = rn_div(theta * theta, 1.f - c);
  const float x0 = (R[0] - c) * b, x1 = (R[4] - c) * b, x2 = (R[8] - c) * b;
  return {(R[7] > R[5] ? 1.f : -1.f) * (x0 > 0.f ? sqrt(x0) : 0.f), (R[2] > R[6] ? 1.f : -1.f) * (x1 > 0.f ? sqrt(x1) : 0.f),
          (R[3] > R[1] ? 1.f : -1.f) * (x2 > 0.f ? sqrt(x2) : 0.f)};
}

// alpha = (t/2) cot(t/2), beta = (1 - alpha) / t^2, dbeta = beta'(t) / t: the
// series, for t below 0.5.
template <class T> __device__ __forceinline__ void log_series(T t, T &alpha, T &beta, T &dbeta) {
  const T t2 = t * t;
  alpha = T(1) - t2 * (T(1) / T(12) + t2 * (T(1) / T(720) + t2 * (T(1) / T(30240) + rn_div_by(t2, T(1209600)))));
  beta = T(1) / T(12) +
         t2 * (T(1) / T(720) + t2 * (T(1) / T(30240) + t2 * (T(1) / T(1209600) + rn_div_by(t2, T(47900160)))));
  dbeta = T(1) / T(360) + t2 * (T(1) / T(7560) + t2 * (T(1) / T(201600) + rn_div_by(t2, T(5987520))));
}
// st, ct: log3_dev's sin t and cos t.
__device__ __forceinline__ void log_coeffs_dev(float t, float st, float ct, float &alpha, float &beta, float &dbeta) {
  if (t < 0.5f) {
    log_series(t, alpha, beta, dbeta);
  } else {
    // two reciprocals (1/t, 1/(1 - cos t)) instead of one division per term
    const float r = rn_rcp(t), u = rn_rcp(1.f - ct), r2 = r * r, hsu = 0.5f * st * u;
    alpha = t * hsu;
    beta = r2 - r * hsu;
    dbeta = -2.f * r2 * r2 + (1.f + st * r) * (0.5f * u) * r2;
  }
}

__device__ __forceinline__ S6<float> log6_dev(const float *R, V3<float> p) {
  float t, st, ct;
  V3<float> w = log3_dev(R, t, st, ct);
  float al, be, db;
  log_coeffs_dev(t, st, ct, al, be, db);
  return {al * p - 0.5f * cross(w, p) + (be * dot(w, p)) * w, w};
}

// Jlog6 (6x6 row-major): [[A, C A], [0, A]], A = alpha I + beta w w^T + [w]x / 2,
// C = dbeta (w.p) w w^T - (t^2 dbeta + 2 beta) p w^T + beta w p^T + beta (w.p) I + [p]x / 2.
// jlog6_blocks gives the 3x3 blocks A and C; jlog6_core the assembled matrix.
template <class T>
__device__ __forceinline__ void jlog6_blocks(V3<T> w, T t, T al, T be, T db, V3<T> p, T *A, T *C) {
  T wv[3] = {w.x, w.y, w.z}, pv[3] = {p.x, p.y, p.z};
  T wp = dot(w, p);
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      A[3 * i + j] = be * wv[i] * wv[j] + (i == j ? al : T(0));
      C[3 * i + j] = db * wp * wv[i] * wv[j] - (t * t * db + T(2) * be) * pv[i] * wv[j] + be * wv[i] * pv[j] +
                     (i == j ? be * wp : T(0));
    }
  A[1] -= T(0.5) * w.z; A[2] += T(0.5) * w.y; A[5] -= T(0.5) * w.x;
  A[3] += T(0.5) * w.z; A[6] -= T(0.5) * w.y; A[7] += T(0.5) * w.x;
  C[1] -= T(0.5) * p.z; C[2] += T(0.5) * p.y; C[5] -= T(0.5) * p.x;
  C[3] += T(0.5) * p.z; C[6] -= T(0.5) * p.y; C[7] += T(0.5) * p.x;
}
__device__ __forceinline__ void jlog6_core(V3<float> w, float t, float al, float be, float db, V3<float> p, float *Jl) {
  float A[9], C[9];
  jlog6_blocks(w, t, al, be, db, p, A, C);
  float CA[9];
  mm(C, A, CA);
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      Jl[i * 6 + j] = A[3 * i + j];
      Jl[i * 6 + 3 + j] = CA[3 * i + j];
      Jl[(3 + i) * 6 + j] = 0.f;
      Jl[(3 + i) * 6 + 3 + j] = A[3 * i + j];
    }
}

__device__ __forceinline__ void jlog6_dev(const float *R, V3<float> p, float *Jl) {
  float t, st, ct;
  V3<float> w = log3_dev(R, t, st, ct);
  float al, be, db;
  log_coeffs_dev(t, st, ct, al, be, db);
  jlog6_core(w, t, al, be, db, p, Jl);
}

// log6 of (R, p) and Jlog6 of its inverse (R^T, -R^T p) from one rotation log:
// log3(R^T) = -log3(R) (the axial vector changes sign exactly, the angle and
// the coefficients are the same; in the branch near pi the signs come from the
// skew part, which also flips, unless two of its entries tie exactly), so this
// equals log6_dev(R, p) and jlog6_dev(R^T, -R^T p) bit for bit.
__device__ __forceinline__ S6<float> log6_jlog6_inv(const float *R, V3<float> p, float *Jl) {
  float t, st, ct;
  V3<float> w = log3_dev(R, t, st, ct);
  float al, be, db;
  log_coeffs_dev(t, st, ct, al, be, db);
  jlog6_core(-1.f * w, t, al, be, db, -1.f * mtv(R, p), Jl);
  return {al * p - 0.5f * cross(w, p) + (be * dot(w, p)) * w, w};
}
// The same with Jlog6(M^-1) as its blocks A, C: Jlog6 v = [A v_l + C (A v_a); A v_a]
// costs 27 products per column instead of 36, and C A is never formed.
__device__ __forceinline__ S6<float> log6_jlog6_inv_blocks(const float *R, V3<float> p, float *A, float *C) {
  float t, st, ct;
  V3<float> w = log3_dev(R, t, st, ct);
  float al, be, db;
  log_coeffs_dev(t, st, ct, al, be, db);
  jlog6_blocks(-1.f * w, t, al, be, db, -1.f * mtv(R, p), A, C);
  return {al * p - 0.5f * cross(w, p) + (be * dot(w, p)) * w, w};
}

// 1 / d as the compiler's FP64 division computes it (hardware reciprocal, two
// Newton steps, one residual correction, the fix-up of zeros, infinities and
// NaN) without that division's scaling, which only matters for pivots beyond
// 2^+-1000: the same bits in 8 instructions instead of 12, in a serial chain.
__device__ __forceinline__ double pivot_rcp(double d) {
  double r = __builtin_amdgcn_rcp(d);
#pragma unroll
  for (int k = 0; k < 3; ++k) r = fma(fma(-d, r, 1.0), r, r);
  return __builtin_amdgcn_div_fixup(r, d, 1.0);
}

// y = (J J^T + damp I)^-1 e by LDL^T of the 6x6 SPD matrix, one reciprocal per
// pivot.
template <class T> __device__ __forceinline__ void ldlt6_solve(T *A, T *y) {
  T inv[6];
  for (int j = 0; j < 6; ++j) {
    T d = A[j * 6 + j];
    for (int k = 0; k < j; ++k) d -= A[j * 6 + k] * A[j * 6 + k] * A[k * 6 + k];
    A[j * 6 + j] = d;
    inv[j] = pivot_rcp(d);
    for (int i = j + 1; i < 6; ++i) {
      T s = A[i * 6 + j];
      for (int k = 0; k < j; ++k) s -= A[i * 6 + k] * A[j * 6 + k] * A[k * 6 + k];
      A[i * 6 + j] = s * inv[j];
    }
  }
  for (int i = 0; i < 6; ++i)
    for (int k = 0; k < i; ++k) y[i] -= A[i * 6 + k] * y[k];
  for (int i = 0; i < 6; ++i) y[i] *= inv[i];
  for (int i = 5; i >= 0; --i)
    for (int k = i + 1; k < 6; ++k) y[i] -= A[k * 6 + i] * y[k];
}

// Target pose p | q (w x y z) -> R, p as Eigen::Quaterniond(w, x, y, z)
// .toRotationMatrix() builds it (pinocchio_model.cpp:255): the quaternion is
// not normalized, so a non-unit q gives (1 - |q|^2) I + |q|^2 R(q / |q|).
template <class T> __device__ __forceinline__ void pose_to_mat(const T *P, T *R, V3<T> &p) {
  const T w = P[3], x = P[4], y = P[5], z = P[6];
  R[0] = T(1) - T(2) * (y * y + z * z); R[1] = T(2) * (x * y - w * z); R[2] = T(2) * (x * z + w * y);
  R[3] = T(2) * (x * y + w * z); R[4] = T(1) - T(2) * (x * x + z * z); R[5] = T(2) * (y * z - w * x);
  R[6] = T(2) * (x * z - w * y); R[7] = T(2) * (y * z + w * x); R[8] = T(1) - T(2) * (x * x + y * y);
  p = {P[0], P[1], P[2]};
}

}  // namespace sapamd
