// One CLIK problem per wavefront in FP64: compute_inverse_kinematics
// (pinocchio_model.cpp:228-300), one configuration per call. Lane k owns chain
// joint k (chains of up to 64 joints), its state in registers and its rotation's
// constants in LDS; what depends on the link's pose alone (the SE(3) log, the
// damped 6x6 solve, the best iterate's bookkeeping) every lane computes for
// itself, so an iteration needs no barrier. Per iteration:
//   FK      a prefix product of the joints' transforms over the lanes (DPP row
//           shifts for chains of up to 16 joints, ds_bpermute past that), the
//           link joint's pose read from its lane into scalars
//   J       each lane's column in the link frame, through Jlog6 of the error
//   J J^T   the columns through LDS, one of the 21 entries per lane, and back
//   solve   L D L^T in every lane
//
// Bound: latency, one wavefront's chain of about 1,100 instructions an
// iteration. An arm of 7 joints and two fingers, about 80 iterations a call: 400 us
// with one block whose thread 0 composed the chain and solved (six barriers an
// iteration), 190 us here (2.25 us an iteration, 2.46 for 12 joints, 3.42 for 40,
// over calls that run to the iteration limit). The rotations' constants stay in
// LDS: in registers the two-finger arm takes 183 us, but 12 joints 200 us instead
// of 193 and 40 joints 341 us instead of 318 (the kernel then needs more than
// the 256 registers an instruction can name).
#include <hip/hip_runtime.h>

#include "call.h"
#include "lanes.h"
#include "launch.h"
#include "se3.h"
#include "spatial.h"

namespace sapamd {

namespace {

using namespace lanes;
using Xd = XfT<double>;
using Vd = V3<double>;

// Value of the lane D below in the 16-lane row, `old` where there is none.
template <int D> __device__ __forceinline__ double row_below(double old, double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x), o = __builtin_bit_cast(uint64_t, old);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)o, (int)(uint32_t)u, 0x110 + D, 0xF, 0xF, false);
  const uint32_t hi =
      (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)(o >> 32), (int)(uint32_t)(u >> 32), 0x110 + D, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double from_lane(double x, int lane) {  // lane: uniform
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// x_k <- x_0 ... x_k over the first nc lanes.
template <int D> __device__ __forceinline__ void row_prefix(Xd &x, int nc) {
  if constexpr (D < 16) {
    if (nc <= D) return;  // uniform
    Xd y;
#pragma unroll
    for (int k = 0; k < 9; ++k) y.R[k] = row_below<D>(k % 4 == 0 ? 1.0 : 0.0, x.R[k]);
    y.p = {row_below<D>(0.0, x.p.x), row_below<D>(0.0, x.p.y), row_below<D>(0.0, x.p.z)};
    x = compose(y, x);
    row_prefix<2 * D>(x, nc);
  }
}
__device__ __forceinline__ void wave_prefix(Xd &x, int nc, int lane) {
  for (int d = 1; d < nc; d *= 2) {  // uniform
    const int src = 4 * (lane >= d ? lane - d : lane);
    Xd y;
#pragma unroll
    for (int k = 0; k < 9; ++k) y.R[k] = bperm(src, x.R[k]);
    y.p = {bperm(src, x.p.x), bperm(src, x.p.y), bperm(src, x.p.z)};
    const Xd z = compose(y, x);
    if (lane >= d) x = z;
  }
}

// 1 / d from the hardware estimate and three Newton steps (d normal).
__device__ __forceinline__ double reciprocal(double d) {
  double r = __builtin_amdgcn_rcp(d);
#pragma unroll
  for (int i = 0; i < 3; ++i) r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return r;
}

// log6_jlog6_inv_blocks (se3.h) with sin and cos of the rotation angle taken
// from its cosine: theta = acos(c), so sin theta = sqrt((1 - c)(1 + c)).
__device__ __forceinline__ S6<double> log_blocks(const double *R, Vd p, double *A, double *C) {
  const double PI = 3.14159265358979323846;
  const double tr = R[0] + R[4] + R[8];
  const double c = tr >= 3.0 ? 1.0 : tr <= -1.0 ? -1.0 : 0.5 * (tr - 1.0);
  const double t = acos(c), st = sqrt((1.0 - c) * (1.0 + c));
  Vd w;
  if (t < PI - 1e-2) {
    const double k = t > 1.220703125e-4 ? t * reciprocal(st) : 1.0;
    w = k * Vd{0.5 * (R[7] - R[5]), 0.5 * (R[2] - R[6]), 0.5 * (R[3] - R[1])};
  } else {
    const double b = t * t / (1.0 - c);
    const double x0 = (R[0] - c) * b, x1 = (R[4] - c) * b, x2 = (R[8] - c) * b;
    w = {(R[7] > R[5] ? 1.0 : -1.0) * (x0 > 0.0 ? sqrt(x0) : 0.0), (R[2] > R[6] ? 1.0 : -1.0) * (x1 > 0.0 ? sqrt(x1) : 0.0),
         (R[3] > R[1] ? 1.0 : -1.0) * (x2 > 0.0 ? sqrt(x2) : 0.0)};
  }
  double al, be, db;
  if (t < 0.5) {
    log_series(t, al, be, db);
  } else {
    const double r = reciprocal(t), u = reciprocal(1.0 - c), r2 = r * r, hsu = 0.5 * st * u;
    al = t * hsu;
    be = r2 - r * hsu;
    db = -2.0 * r2 * r2 + (1.0 + st * r) * (0.5 * u) * r2;
  }
  jlog6_blocks(-1.0 * w, t, al, be, db, -1.0 * mtv(R, p), A, C);
  return {al * p - 0.5 * cross(w, p) + (be * dot(w, p)) * w, w};
}

// y = S^-1 y by LDL^T, S the symmetric 6x6 matrix with lower triangle s (row by row).
__device__ __forceinline__ void solve6(double (&s)[21], double *y) {
  double d[6], inv[6], l[6][6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    double dj = s[j * (j + 1) / 2 + j], ld[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
      if (k < j) {
        ld[k] = l[j][k] * d[k];
        dj -= l[j][k] * ld[k];
      }
    d[j] = dj;
    inv[j] = reciprocal(dj);
#pragma unroll
    for (int i = 0; i < 6; ++i)
      if (i > j) {
        double v = s[i * (i + 1) / 2 + j];
#pragma unroll
        for (int k = 0; k < 6; ++k)
          if (k < j) v -= l[i][k] * ld[k];
        l[i][j] = v * inv[j];
      }
  }
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int k = 0; k < 6; ++k)
      if (k < i) y[i] -= l[i][k] * y[k];
#pragma unroll
  for (int i = 0; i < 6; ++i) y[i] *= inv[i];
#pragma unroll
  for (int i = 5; i >= 0; --i)
#pragma unroll
    for (int k = 0; k < 6; ++k)
      if (k > i) y[i] -= l[k][i] * y[k];
}

// Target pose p | q wxyz.
struct CallPose {
  double x[7];
};

template <bool ROW>
__global__ __launch_bounds__(64) void k_clik_wave(CallModel m, ClikParams P, CallPose T, CallIn<2> in,
                                                  double *__restrict__ q_out, double *__restrict__ err_out,
                                                  int32_t *__restrict__ success, int32_t *__restrict__ iters) {
  __shared__ __align__(16) double s_J[64 * 6], s_S[22], s_rec[27][64];
  __shared__ int s_chain[64];
  const ModelTable<double> *const M = m.tab;
  const int lane = threadIdx.x, nc = P.nchain, nj = m.nj;
  const bool valid = lane < nc;
  const JointRec<double> *JR = joints_of(M);
  const int joint = valid ? P.chain[lane] : 0;
  const JointRec<double> &J = JR[joint];  // read by valid lanes only
  // this lane's joint: R(q) = A + sin q B + (1 - cos q) C, p(q) = p + q ap
  // (identity and a zero column past the chain end)
  const int kind = valid ? J.kind : KIND_REVOLUTE;
  const bool slides = kind == KIND_PRISMATIC;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    s_rec[k][lane] = valid ? J.A[k] : k % 4 == 0 ? 1.0 : 0.0;
    s_rec[9 + k][lane] = valid ? J.Bq[k] : 0.0;  // zero for prismatic joints
    s_rec[18 + k][lane] = valid ? J.Cq[k] : 0.0;
  }
  const Vd zero = {0.0, 0.0, 0.0};
  const Vd pj = valid ? load3(J.p) : zero, ap = valid && slides ? load3(J.ap) : zero;
  const Vd axis = valid ? load3(J.axis) : zero;
  const int u = valid ? J.vuser : 0;
  double q = valid ? in.x[0][joint] : 0.0, qbest = q;
  const double mask = valid ? in.x[1][joint] : 1.0;
  // desired pose of the link's joint frame: oMdes = target * link2joint^-1
  const LinkRec<double> &Lk = links_of(M)[P.link];
  double Rt[9], Rd[9];
  Vd pt;
  pose_to_mat(T.x, Rt, pt);
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      Rd[3 * i + j] = Rt[3 * i] * Lk.R[3 * j] + Rt[3 * i + 1] * Lk.R[3 * j + 1] + Rt[3 * i + 2] * Lk.R[3 * j + 2];
  const Vd pd = pt - mv(Rd, load3(Lk.p));
  // lane t < 21 sums entry (row, column) of the lower triangle of J J^T
  int er = 0;
  while ((er + 1) * (er + 2) / 2 <= lane && er < 5) ++er;
  const int ec = lane - er * (er + 1) / 2 < 6 ? lane - er * (er + 1) / 2 : 0;

  // errors are compared by their squares (eps^2 kept above zero for a positive eps)
  const double eps2 = P.eps > 0.0 ? fmax(P.eps * P.eps, 4.9406564584124654e-324) : 0.0;
  double min2 = 1e20, best[6] = {0, 0, 0, 0, 0, 0};
  bool ok = false;
  int it = 0;
  for (;; ++it) {
    double s, c;
    sincos(slides ? 0.0 : q, &s, &c);
    const double omc = 1.0 - c;
    Xd X;
#pragma unroll
    for (int k = 0; k < 9; ++k) X.R[k] = s_rec[k][lane] + s * s_rec[9 + k][lane] + omc * s_rec[18 + k][lane];
    X.p = pj + q * ap;
    if constexpr (ROW) row_prefix<1>(X, nc);
    else wave_prefix(X, nc, lane);
    Xd E = identity_xf<double>();
    if (nc > 0) {
#pragma unroll
      for (int k = 0; k < 9; ++k) E.R[k] = from_lane(X.R[k], nc - 1);
      E.p = {from_lane(X.p.x, nc - 1), from_lane(X.p.y, nc - 1), from_lane(X.p.z, nc - 1)};
    }
    // iMd = oMj^-1 oMdes, its log and Jlog6 of its inverse
    double Ri[9], Ja[9], Jc[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) Ri[3 * i + j] = E.R[i] * Rd[j] + E.R[3 + i] * Rd[3 + j] + E.R[6 + i] * Rd[6 + j];
    const S6<double> e = log_blocks(Ri, mtv(E.R, pd - E.p), Ja, Jc);
    double ev[6];
    vec_of(e, ev);
    const double e2 = dot6(e, e);
    if (__builtin_amdgcn_readfirstlane(e2 < min2)) {  // the same in every lane
      min2 = e2;
      qbest = q;
#pragma unroll
      for (int r = 0; r < 6; ++r) best[r] = ev[r];
    }
    ok = __builtin_amdgcn_readfirstlane(e2 < eps2);
    if (ok || it >= P.max_iter) break;

    // this lane's column in the link joint's frame, through Jlog6
    const Vd aw = mv(X.R, axis);
    const Vd lin = slides ? aw : cross(X.p - E.p, aw);
    const Vd al = slides ? zero : mtv(E.R, aw);
    const Vd ju = mv(Ja, al), top = mv(Ja, mtv(E.R, lin)) + mv(Jc, ju);
    double Jk[6] = {top.x, top.y, top.z, ju.x, ju.y, ju.z};
#pragma unroll
    for (int r = 0; r < 6; ++r) {
      Jk[r] *= -mask;
      s_J[lane * 6 + r] = Jk[r];
    }
    wave_sync();
    if (lane < 21) {
      double acc = er == ec ? P.damp : 0.0;
      for (int k0 = 0; k0 < nc; k0 += 8)  // columns past the chain end are zero
#pragma unroll
        for (int k = k0; k < k0 + 8; ++k) acc += s_J[k * 6 + er] * s_J[k * 6 + ec];
      s_S[lane] = acc;
    }
    wave_sync();
    double S[21], y[6];
#pragma unroll
    for (int i = 0; i < 21; ++i) S[i] = s_S[i];
#pragma unroll
    for (int r = 0; r < 6; ++r) y[r] = ev[r];
    solve6(S, y);
    double v = 0.0;
#pragma unroll
    for (int r = 0; r < 6; ++r) v -= Jk[r] * y[r];
    if (valid) q += v * P.dt;
  }
  // result: chain dofs from the best iterate, the rest from q0; every
  // continuous dof wrapped by atan2 (posP2S over the whole configuration,
  // pinocchio_model.cpp:87,299)
  s_chain[lane] = 0;
  wave_sync();
  if (valid) s_chain[joint] = 1;
  wave_sync();
  const auto wrapped = [](double v, int kind) {
    if (kind != KIND_CONTINUOUS) return v;
    double s, c;
    sincos(v, &s, &c);
    return atan2(s, c);
  };
  if (valid) q_out[u] = wrapped(qbest, kind);
  if (lane < nj && !s_chain[lane]) {
    const int w = JR[lane].vuser;
    q_out[w] = wrapped(in.x[0][lane], JR[lane].kind);
  }
  if (lane == 0) {
    success[0] = ok ? 1 : 0;
#pragma unroll
    for (int r = 0; r < 6; ++r) err_out[r] = best[r];
    iters[0] = it;
  }
  call_done(m);
}

}  // namespace

hipError_t launch_clik_wave(const CallModel &m, const ClikParams &P, const double *target, const CallIn<2> &q0_mask,
                            double *q_out, double *err, int32_t *success, int32_t *iters, hipStream_t s) {
  if (m.nj > 64 || P.nchain > 64) return hipErrorNotSupported;
  CallPose T;
  for (int i = 0; i < 7; ++i) T.x[i] = target[i];
  if (P.nchain <= 16)
    hipLaunchKernelGGL(k_clik_wave<true>, dim3(1), dim3(64), 0, s, m, P, T, q0_mask, q_out, err, success, iters);
  else
    hipLaunchKernelGGL(k_clik_wave<false>, dim3(1), dim3(64), 0, s, m, P, T, q0_mask, q_out, err, success, iters);
  return hipGetLastError();
}

}  // namespace sapamd
