// The per-call methods (one configuration, FP64, the reference's use): one
// wavefront per call, lane j owning joint j of the depth-first order (trees of up
// to 64 joints), inputs handed over as kernel arguments and results written to
// the model's pinned per-call buffer.
//   X, v, a      root to joint: pointer jumping with ds_bpermute, log2(depth) rounds
//   F, Ic, ABA   leaves to root: level by level through LDS, a joint adding its
//                children's values (their lanes are j + 1 and then each
//                sibling's end, the subtrees being contiguous)
//   outputs      (link, dof) and (dof, dof) entries over all 64 lanes, from the
//                columns and forces in LDS
// The loops over rounds, levels and entries stay rolled: a call runs its code
// once, from a cold instruction cache, so short code is fast code.
//
// Bound: latency (an empty launch is 1.7 us). Kernel time in us for a 9-joint arm
// / a 30-joint tree, and before with a block whose thread 0 ran the compositions,
// sums and the ABA recursion: poses 5.4 / 5.9 (8.4 / 13.6), with all link
// Jacobians 6.2 / 13.3 (9.7 / 24.5), M 6.8 / 10.8 (10.8 / 24.6), C 9.3 / 15.9
// (13.5 / 31.7), inverse dynamics 7.1 / 8.4 (13.2 / 32.4), forward dynamics
// 11.8 / 15.2 (23.2 / 60.8).
#include <hip/hip_runtime.h>

#include "call.h"
#include "lanes.h"
#include "launch.h"
#include "se3.h"
#include "spatial.h"
#include "tree.h"

namespace sapamd {

namespace {

using namespace lanes;
using Xd = XfT<double>;
using Vd = V3<double>;
using Sd = S6<double>;

// This lane's joint, its constants in registers (one round of loads), and its
// place in the tree. Lanes past the last joint hold the identity and zeros.
struct CallJoint {
  JointRec<double> J;
  int lane, parent, size, depth, u;
  bool valid, slides;
};

template <bool INERTIA> __device__ __forceinline__ CallJoint call_joint(const ModelTable<double> *M, int nj) {
  CallJoint c;
  c.lane = threadIdx.x;
  c.valid = c.lane < nj;
  c.parent = -1;
  c.size = c.depth = c.u = 0;
  c.slides = false;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    c.J.A[k] = k % 4 == 0 ? 1.0 : 0.0;
    c.J.Bq[k] = c.J.Cq[k] = 0.0;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) c.J.p[k] = c.J.ap[k] = c.J.axis[k] = 0.0;
  if (c.valid) {
    const JointRec<double> &J = joints_of(M)[c.lane];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      c.J.A[k] = J.A[k];
      c.J.Bq[k] = J.Bq[k];
      c.J.Cq[k] = J.Cq[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      c.J.p[k] = J.p[k];
      c.J.ap[k] = J.ap[k];
      c.J.axis[k] = J.axis[k];
      if (INERTIA) c.J.c[k] = J.c[k];
    }
    if (INERTIA) {
      c.J.m = J.m;
#pragma unroll
      for (int k = 0; k < 6; ++k) c.J.Ic[k] = J.Ic[k];
    }
    c.parent = J.parent;
    c.size = J.subtree;
    c.depth = J.depth;
    c.u = J.vuser;
    c.slides = J.kind == KIND_PRISMATIC;
  }
  return c;
}

// f(y, has) for each pointer-jumping round, y(x) giving the value of x at the
// current ancestor (any lane's where there is none).
template <class F> __device__ __forceinline__ void to_root(const CallJoint &c, int max_depth, F &&f) {
  int a = c.parent;
  for (int reach = 1; reach < max_depth; reach *= 2) {  // uniform
    const bool has = a >= 0;
    const int src = has ? 4 * a : 0;
    f([&](double x) { return bperm(src, x); }, has);
    const int next = __builtin_amdgcn_ds_bpermute(src, a);
    a = has ? next : -1;
  }
}

__device__ __forceinline__ Xd world_pose(const CallJoint &c, int max_depth, double q) {
  Xd X;
  double s, co;
  sincos(c.slides ? 0.0 : q, &s, &co);
  const double omc = 1.0 - co;
#pragma unroll
  for (int k = 0; k < 9; ++k) X.R[k] = c.J.A[k] + s * c.J.Bq[k] + omc * c.J.Cq[k];  // B = C = 0: prismatic
  X.p = load3(c.J.p) + (c.slides ? q : 0.0) * load3(c.J.ap);
  to_root(c, max_depth, [&](auto &&at, bool has) {
    Xd y;
#pragma unroll
    for (int k = 0; k < 9; ++k) y.R[k] = at(X.R[k]);
    y.p = {at(X.p.x), at(X.p.y), at(X.p.z)};
    const Xd z = compose(y, X);
    if (has) X = z;
  });
  return X;
}
// x_j <- sum of x over joint j and its ancestors
__device__ __forceinline__ void path_sum(const CallJoint &c, int max_depth, Sd &x) {
  to_root(c, max_depth, [&](auto &&at, bool has) {
    const Sd y = {{at(x.l.x), at(x.l.y), at(x.l.z)}, {at(x.a.x), at(x.a.y), at(x.a.z)}};
    if (has) x = x + y;
  });
}

// One level of a leaves-to-root pass: joints at `depth` offer x, their parents
// add it.
template <int N>
__device__ __forceinline__ void level_up(const CallJoint &c, int depth, double (&x)[N], double (*buf)[64],
                                         const int *s_size) {
  if (c.depth == depth) {
#pragma unroll
    for (int i = 0; i < N; ++i) buf[i][c.lane] = x[i];
  }
  wave_sync();
  if (c.valid && c.depth == depth - 1)
    for (int k = c.lane + 1; k < c.lane + c.size; k += s_size[k]) {
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] += buf[i][k];
    }
  wave_sync();
}
template <int N>
__device__ __forceinline__ void subtree_sum(const CallJoint &c, int max_depth, double (&x)[N], double (*buf)[64],
                                            const int *s_size) {
  for (int d = max_depth; d > 1; --d) level_up(c, d, x, buf, s_size);
}

__device__ __forceinline__ Sd column(const CallJoint &c, const Xd &X) {
  const Vd a = mv(X.R, load3(c.J.axis));  // zero past the last joint
  return c.slides ? Sd{a, {0.0, 0.0, 0.0}} : Sd{cross(X.p, a), a};
}
__device__ __forceinline__ void put6(double (*buf)[64], int lane, const Sd &x) {
  buf[0][lane] = x.l.x; buf[1][lane] = x.l.y; buf[2][lane] = x.l.z;
  buf[3][lane] = x.a.x; buf[4][lane] = x.a.y; buf[5][lane] = x.a.z;
}
__device__ __forceinline__ Sd get6(const double (*buf)[64], int lane) {
  return {{buf[0][lane], buf[1][lane], buf[2][lane]}, {buf[3][lane], buf[4][lane], buf[5][lane]}};
}

// Link poses, every link's Jacobians, or one link's body-frame Jacobian (link >= 0).
struct CallKinematics {
  double *poses, *jw, *jl;  // (L, 7), (L, 6, nv) each; NULL = not wanted
  int link;                 // -1 = every link
};
__global__ __launch_bounds__(64) void k_call_kinematics(CallModel m, CallIn<1> in, CallKinematics out) {
  __shared__ double s_X[12][64], s_col[6][64], s_link[12][64];
  __shared__ int s_joint[64], s_end[64], s_on[64];  // joint of a dof; end of a joint's subtree; a link's joint
  const ModelTable<double> *const M = m.tab;
  const int nj = m.nj, max_depth = m.max_depth;
  const CallJoint c = call_joint<false>(M, nj);
  const int lane = c.lane, nv = nj, nlinks = m.nlinks;
  const Xd X = world_pose(c, max_depth, c.valid ? in.x[0][c.lane] : 0.0);
#pragma unroll
  for (int k = 0; k < 9; ++k) s_X[k][lane] = X.R[k];
  s_X[9][lane] = X.p.x; s_X[10][lane] = X.p.y; s_X[11][lane] = X.p.z;
  put6(s_col, lane, column(c, X));
  if (c.valid) {
    s_joint[c.u] = lane;
    s_end[lane] = lane + c.size;
  }
  wave_sync();
  const int first = out.link < 0 ? 0 : out.link, end = out.link < 0 ? nlinks : out.link + 1;
  for (int l0 = first; l0 < end; l0 += 64) {
    const int n = end - l0 < 64 ? end - l0 : 64;
    if (lane < n) {
      const LinkRec<double> &K = links_of(M)[l0 + lane];
      double R[9];
      Vd p = load3(K.p);
#pragma unroll
      for (int k = 0; k < 9; ++k) R[k] = K.R[k];
      if (K.joint >= 0) {
        double Rj[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) Rj[k] = s_X[k][K.joint];
        mm(Rj, K.R, R);
        p = mv(Rj, p) + Vd{s_X[9][K.joint], s_X[10][K.joint], s_X[11][K.joint]};
      }
#pragma unroll
      for (int k = 0; k < 9; ++k) s_link[k][lane] = R[k];
      s_link[9][lane] = p.x; s_link[10][lane] = p.y; s_link[11][lane] = p.z;
      s_on[lane] = K.joint;
      if (out.poses) {
        double *P = out.poses + (int64_t)(l0 + lane) * 7;
        P[0] = p.x; P[1] = p.y; P[2] = p.z;
        quat_of(R, P + 3);
      }
    }
    wave_sync();
    if (out.jl)
      for (int i = lane; i < n * nv; i += 64) {
        const int l = i / nv, u = i - l * nv;
        const int j = s_joint[u], jl = s_on[l];
        Sd cw = zero6<double>(), cl = zero6<double>();
        if (j <= jl && jl < s_end[j]) {  // the joint carries the link
          double R[9];
#pragma unroll
          for (int k = 0; k < 9; ++k) R[k] = s_link[k][l];
          cw = get6(s_col, j);
          cl = to_local(R, Vd{s_link[9][l], s_link[10][l], s_link[11][l]}, cw);
        }
        const int64_t at = (out.link < 0 ? (int64_t)(l0 + l) * 6 * nv : 0) + u;
        double *Jl = out.jl + at;
        Jl[0] = cl.l.x; Jl[nv] = cl.l.y; Jl[2 * nv] = cl.l.z;
        Jl[3 * nv] = cl.a.x; Jl[4 * nv] = cl.a.y; Jl[5 * nv] = cl.a.z;
        if (out.jw) {
          double *Jw = out.jw + at;
          Jw[0] = cw.l.x; Jw[nv] = cw.l.y; Jw[2 * nv] = cw.l.z;
          Jw[3 * nv] = cw.a.x; Jw[4 * nv] = cw.a.y; Jw[5 * nv] = cw.a.z;
        }
      }
    wave_sync();
  }
  call_done(m);
}

__device__ __forceinline__ Sd gravity_of(const ModelTable<double> *M) {
  return {{-M->gravity[0], -M->gravity[1], -M->gravity[2]}, {0.0, 0.0, 0.0}};
}

// Inverse dynamics: tau (nv).
__global__ __launch_bounds__(64) void k_call_rnea(CallModel m, CallIn<3> in, double *__restrict__ tau) {
  __shared__ double s_buf[6][64];
  __shared__ int s_size[64];
  const ModelTable<double> *const M = m.tab;
  const int nj = m.nj, max_depth = m.max_depth;
  const CallJoint c = call_joint<true>(M, nj);
  const double qj = c.valid ? in.x[0][c.lane] : 0.0, v1 = c.valid ? in.x[1][c.lane] : 0.0, a1 = c.valid ? in.x[2][c.lane] : 0.0;
  s_size[c.lane] = c.size;
  const Xd X = world_pose(c, max_depth, qj);
  const Sd col = column(c, X);
  Sd v = v1 * col;
  path_sum(c, max_depth, v);
  Sd a = a1 * col + v1 * crossm(v, col);
  path_sum(c, max_depth, a);
  a = a + gravity_of(M);
  double f[6] = {0, 0, 0, 0, 0, 0};
  if (c.valid) {
    const WInertia<double> Y = world_inertia(c.J, X.R, X.p);
    vec_of(inertia_apply(Y, a) + crossf(v, inertia_apply(Y, v)), f);
  }
  subtree_sum(c, max_depth, f, s_buf, s_size);
  if (c.valid) tau[c.u] = dot6(col, Sd{{f[0], f[1], f[2]}, {f[3], f[4], f[5]}});
  call_done(m);
}

// Mass matrix (nv, nv): M_ij = col_a . (Ic_d col_d), a the ancestor-or-self of d.
__global__ __launch_bounds__(64) void k_call_mass(CallModel m, CallIn<1> in, double *__restrict__ out) {
  __shared__ double s_buf[10][64], s_col[6][64];
  __shared__ int s_size[64], s_joint[64];
  const ModelTable<double> *const M = m.tab;
  const int nj = m.nj, max_depth = m.max_depth;
  const CallJoint c = call_joint<true>(M, nj);
  const int nv = nj;
  s_size[c.lane] = c.size;
  if (c.valid) s_joint[c.u] = c.lane;
  const Xd X = world_pose(c, max_depth, c.valid ? in.x[0][c.lane] : 0.0);
  const Sd col = column(c, X);
  double y[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (c.valid) {
    const AInertia<double> Y = additive(world_inertia(c.J, X.R, X.p));
    y[0] = Y.m; y[1] = Y.h.x; y[2] = Y.h.y; y[3] = Y.h.z;
#pragma unroll
    for (int k = 0; k < 6; ++k) y[4 + k] = Y.I[k];
  }
  subtree_sum(c, max_depth, y, s_buf, s_size);
  const AInertia<double> Ic = {y[0], {y[1], y[2], y[3]}, {y[4], y[5], y[6], y[7], y[8], y[9]}};
  put6(s_col, c.lane, col);
  put6(s_buf, c.lane, apply(Ic, col));
  wave_sync();
  for (int e = c.lane; e < nv * nv; e += 64) {
    const int r = e / nv, i = s_joint[r], j = s_joint[e - r * nv];
    const int a = i < j ? i : j, d = i < j ? j : i;
    out[e] = d < a + s_size[a] ? dot6(get6(s_col, a), get6(s_buf, d)) : 0.0;
  }
  call_done(m);
}

// Coriolis matrix (nv, nv), with the 12-number B of kernels_matrices.hip.
__global__ __launch_bounds__(64) void k_call_coriolis(CallModel m, CallIn<2> in, double *__restrict__ out) {
  __shared__ double s_buf[27][64];
  __shared__ int s_size[64], s_joint[64];
  const ModelTable<double> *const M = m.tab;
  const int nj = m.nj, max_depth = m.max_depth;
  const CallJoint c = call_joint<true>(M, nj);
  const int nv = nj;
  const double qj = c.valid ? in.x[0][c.lane] : 0.0, v1 = c.valid ? in.x[1][c.lane] : 0.0;
  s_size[c.lane] = c.size;
  if (c.valid) s_joint[c.u] = c.lane;
  const Xd X = world_pose(c, max_depth, qj);
  const Sd col = column(c, X);
  Sd v = v1 * col;
  path_sum(c, max_depth, v);
  const Sd dcol = crossm(v, col);
  double x[22];
  if (c.valid) {
    coriolis_terms(additive(world_inertia(c.J, X.R, X.p)), v, x);
  } else {
#pragma unroll
    for (int i = 0; i < 22; ++i) x[i] = 0.0;
  }
  subtree_sum(c, max_depth, x, s_buf, s_size);
  Sd F1, G;
  Vd H;
  coriolis_forces(x, col, dcol, F1, G, H);
  put6(s_buf, c.lane, col);
  put6(s_buf + 6, c.lane, dcol);
  put6(s_buf + 12, c.lane, F1);
  put6(s_buf + 18, c.lane, G);
  s_buf[24][c.lane] = H.x; s_buf[25][c.lane] = H.y; s_buf[26][c.lane] = H.z;
  wave_sync();
  for (int e = c.lane; e < nv * nv; e += 64) {
    const int rr = e / nv, r = s_joint[rr], k = s_joint[e - rr * nv];
    double val = 0.0;
    if (r <= k && k < r + s_size[r]) {  // r ancestor-or-self of k
      val = dot6(get6(s_buf, r), get6(s_buf + 12, k));
    } else if (k < r && r < k + s_size[k]) {  // k strict ancestor of r
      val = dot6(get6(s_buf + 18, r), get6(s_buf + 6, k)) +
            dot(Vd{s_buf[24][r], s_buf[25][r], s_buf[26][r]}, Vd{s_buf[3][k], s_buf[4][k], s_buf[5][k]});
    }
    out[e] = val;
  }
  call_done(m);
}

// Forward dynamics by the articulated-body recursion in the world frame: every
// joint of a level eliminates its own axis (U = IA col, D = col . U), offers its
// parent Ia = IA - U U^T / D (symmetric, 21 numbers) and pa, and the levels are
// walked back to the leaves for the accelerations.
__global__ __launch_bounds__(64) void k_call_aba(CallModel m, CallIn<3> in, double *__restrict__ out) {
  __shared__ double s_buf[27][64];
  __shared__ int s_size[64];
  const ModelTable<double> *const M = m.tab;
  const int nj = m.nj, max_depth = m.max_depth;
  const CallJoint c = call_joint<true>(M, nj);
  const double qj = c.valid ? in.x[0][c.lane] : 0.0, v1 = c.valid ? in.x[1][c.lane] : 0.0, t1 = c.valid ? in.x[2][c.lane] : 0.0;
  s_size[c.lane] = c.size;
  const Xd X = world_pose(c, max_depth, qj);
  const Sd col = column(c, X);
  Sd v = v1 * col;
  path_sum(c, max_depth, v);
  const Sd cb = v1 * crossm(v, col);
  // x: the lower triangle of IA (row by row), then pA
  double x[27], s[6], U[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < 27; ++i) x[i] = 0.0;
  vec_of(col, s);
  if (c.valid) {
    const WInertia<double> Y = world_inertia(c.J, X.R, X.p);
    const AInertia<double> A = additive(Y);
    // [[m 1, -[h]x], [[h]x, I_O]]
    x[0] = x[2] = x[5] = A.m;
    x[7] = -A.h.z; x[8] = A.h.y;
    x[10] = A.h.z; x[12] = -A.h.x;
    x[15] = -A.h.y; x[16] = A.h.x;
    x[9] = A.I[0]; x[13] = A.I[1]; x[14] = A.I[3];
    x[18] = A.I[2]; x[19] = A.I[4]; x[20] = A.I[5];
    vec_of(crossf(v, inertia_apply(Y, v)), x + 21);
  }
  double invD = 0.0, uu = 0.0;
  for (int d = max_depth; d >= 1; --d) {
    double keep[27];
    if (c.depth == d) {
      double D = 0.0;
#pragma unroll
      for (int r = 0; r < 6; ++r) {
        U[r] = 0.0;
#pragma unroll
        for (int k = 0; k < 6; ++k) U[r] += x[r >= k ? r * (r + 1) / 2 + k : k * (k + 1) / 2 + r] * s[k];
      }
#pragma unroll
      for (int r = 0; r < 6; ++r) D += s[r] * U[r];
      uu = t1;
#pragma unroll
      for (int r = 0; r < 6; ++r) uu -= s[r] * x[21 + r];
      invD = 1.0 / D;
    }
    if (d == 1) break;  // uniform: the root joints have no parent
    if (c.depth == d) {
      double cv[6];
      vec_of(cb, cv);
#pragma unroll
      for (int r = 0; r < 6; ++r)
#pragma unroll
        for (int k = 0; k <= r; ++k) keep[r * (r + 1) / 2 + k] = x[r * (r + 1) / 2 + k] - U[r] * U[k] * invD;
#pragma unroll
      for (int r = 0; r < 6; ++r) {
        double t = x[21 + r] + uu * invD * U[r];
#pragma unroll
        for (int k = 0; k < 6; ++k) t += keep[r >= k ? r * (r + 1) / 2 + k : k * (k + 1) / 2 + r] * cv[k];
        keep[21 + r] = t;
      }
#pragma unroll
      for (int i = 0; i < 27; ++i) x[i] = keep[i];
    }
    level_up(c, d, x, s_buf, s_size);
  }
  Sd a = gravity_of(M);  // the parent's acceleration, then this joint's
  const int src = 4 * (c.parent >= 0 ? c.parent : 0);
  for (int d = 1; d <= max_depth; ++d) {
    const Sd ap = {{bperm(src, a.l.x), bperm(src, a.l.y), bperm(src, a.l.z)},
                   {bperm(src, a.a.x), bperm(src, a.a.y), bperm(src, a.a.z)}};
    if (c.depth == d) {
      a = (d > 1 ? ap : a) + cb;
      const double t = (uu - dot6(Sd{{U[0], U[1], U[2]}, {U[3], U[4], U[5]}}, a)) * invD;
      out[c.u] = t;
      a = a + t * col;
    }
  }
  call_done(m);
}

}  // namespace

hipError_t launch_call_kinematics(const CallModel &m, const CallIn<1> &q, double *poses, double *jw, double *jl,
                                  int link, hipStream_t s) {
  if (m.nj > 64) return hipErrorNotSupported;
  hipLaunchKernelGGL(k_call_kinematics, dim3(1), dim3(64), 0, s, m, q, CallKinematics{poses, jw, jl, link});
  return hipGetLastError();
}
hipError_t launch_call_rnea(const CallModel &m, const CallIn<3> &q_qd_qdd, double *tau, hipStream_t s) {
  if (m.nj > 64) return hipErrorNotSupported;
  hipLaunchKernelGGL(k_call_rnea, dim3(1), dim3(64), 0, s, m, q_qd_qdd, tau);
  return hipGetLastError();
}
hipError_t launch_call_mass(const CallModel &m, const CallIn<1> &q, double *out, hipStream_t s) {
  if (m.nj > 64) return hipErrorNotSupported;
  hipLaunchKernelGGL(k_call_mass, dim3(1), dim3(64), 0, s, m, q, out);
  return hipGetLastError();
}
hipError_t launch_call_coriolis(const CallModel &m, const CallIn<2> &q_qd, double *out, hipStream_t s) {
  if (m.nj > 64) return hipErrorNotSupported;
  hipLaunchKernelGGL(k_call_coriolis, dim3(1), dim3(64), 0, s, m, q_qd, out);
  return hipGetLastError();
}
hipError_t launch_call_aba(const CallModel &m, const CallIn<3> &q_qd_tau, double *out, hipStream_t s) {
  if (m.nj > 64) return hipErrorNotSupported;
  hipLaunchKernelGGL(k_call_aba, dim3(1), dim3(64), 0, s, m, q_qd_tau, out);
  return hipGetLastError();
}

}  // namespace sapamd
