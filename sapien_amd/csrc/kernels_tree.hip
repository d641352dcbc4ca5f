// Lanes-per-joint kernels for kinematic trees (FP32), and the heterogeneous
// launch that runs several trees in one grid.
//
// An environment occupies as many lanes as it has joints, or a group of 8, 16
// or 32; lane j owns joint j of the depth-first (preorder) joint order. Two tree
// scans replace the serial sweeps:
//  * root-to-joint prefix (FK products, velocities, accelerations): pointer
//    jumping over the precomputed 2^k-th ancestors, x_j <- x_anc_k(j) (+) x_j
//    for k = 0 .. log2(depth), exchanging registers with ds_bpermute;
//  * subtree sums (forces, composite inertias): in preorder the subtree of j is
//    the lane range [j, j + size_j). Doubling builds block sums
//    B_k[j] = sum of 2^k lanes from j, and F_j adds the blocks of the binary
//    decomposition of size_j. Exact, without prefix differences (no cancellation).
// CRBA: M_ij = col_i . (Yc_j col_j) for i an ancestor-or-self of j, zero between
// joints of different branches.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lanes.h"
#include "launch.h"
#include "spatial.h"
#include "tree.h"

namespace sapamd {

namespace {

using namespace lanes;

constexpr int kMaxTreeJoints = 32;
constexpr int kTreeTableWords4 = (int)((kHeaderBytes + sizeof(JointRec<float>) * kMaxTreeJoints) / 16);

struct TreeIO {
  const float *q, *qd, *qdd;
  float *poses, *J, *tau, *M;
  TreePacking pack;
  // row strides in elements (0 = contiguous: nv, L * 7 and 7)
  int64_t ld_q = 0, ld_qd = 0, ld_qdd = 0, ld_tau = 0, pose_env = 0, pose_link = 0;
};

// Wavefronts per block of k_tree_fused, and the dynamic LDS per wavefront of a
// launch that computes M (its columns and its environments' matrices, up to 18 KB
// for one environment of 64 joints).
constexpr int tree_waves(int width) { return width > 32 ? 2 : 4; }
int tree_wave_floats(const TreePacking &p) {
  if (p.dense) return 64 * 12;
  return AncestorRows<1>::kFloats + ((p.per_wave * p.nj * p.nj + 3) & ~3);
}

// Element offset of row env0 + row (row < 64) of an array with rows every ld
// elements (0 = width): the product with the wavefront's env0 stays scalar.
__device__ __forceinline__ int64_t row_at(int64_t env0, int row, int64_t ld, int width) {
  const int64_t w = ld ? ld : width;
  return env0 * w + (w < (1 << 24) ? (int64_t)__umul24(row, (int)w) : row * w);
}

// One environment per `stride` lanes (lane j owns joint j), per_wave of them
// back to back in the wavefront; M is the LDS copy of the model table, Mg the
// table in memory (its header is read as scalars); lds is the wavefront's part of
// the dynamic LDS (with KF_CRBA); wave is its index within the model's batch.
//
// Bound: the LDS pipe. A ds_bpermute of a wavefront takes it 6.9 cycles and an
// environment of 9 joints needs 105 of them, beside which the records read from
// the staged table and, at 4 cycles a SIMD, 780 VALU instructions have to fit. So
// what pays is a wavefront's exchanges serving more environments: 7 of 9 joints
// instead of 4 in groups of 16 lanes, and only the pointer-jumping rounds that
// the deepest joint needs. 524287 environments of that tree, a call: 212 us in
// 16-lane groups, 135 us packed, 126 with the subtree sums' first two rounds as
// wavefront shifts (337 MB, 72 us at a copy's rate): the LDS pipe is busy for
// 110 us of it with 131 exchanges a wavefront, the vector units for 93. Poses
// and Jacobians staged through LDS for whole-sector stores: 155 us (packed then:
// 138).
template <int G, bool SPARE>
__device__ __forceinline__ void tree_body(const ModelTable<float> *M, const ModelTable<float> *__restrict__ Mg,
                                          int64_t B, int64_t wave, int flags, const TreeIO &io, float *lds) {
  const int nj = io.pack.nj, nv = nj, L = io.pack.nlinks;  // one dof per joint
  PackedTree<G, SPARE> T;
  T.place(io.pack);
  const int g = T.g;
  const int64_t env0 = wave * io.pack.per_wave;
  if (env0 >= B) return;  // a wavefront of the last block
  const int left = (int)(B - env0 < io.pack.per_wave ? B - env0 : io.pack.per_wave);
  const bool live = T.slot < left;
  const int row = live ? T.slot : left - 1;  // this lane's environment after env0 (its last one stands in)
  const bool dyn = flags & KF_RNEA;
  const bool valid = T.slot < io.pack.per_wave && g < nj;
  const JointRec<float> &J = *reinterpret_cast<const JointRec<float> *>(
      reinterpret_cast<const char *>(joints_of(M)) + __umul24(valid ? g : nj - 1, (int)sizeof(JointRec<float>)));
  T.bind(J, valid);

  // dofs: lane g loads user dof g, then the joint -> dof permutation via bpermute
  const int gc = g < nv ? g : nv - 1;
  float qu = io.q[row_at(env0, row, io.ld_q, nv) + gc], qdu = io.qd[row_at(env0, row, io.ld_qd, nv) + gc],
        qddu = io.qdd[row_at(env0, row, io.ld_qdd, nv) + gc];
  const int src = valid ? T.base4 + 4 * J.vuser : 0;
  float qj = bperm(src, qu), qdj = bperm(src, qdu), qddj = bperm(src, qddu);
  if (!valid) qj = qdj = qddj = 0.f;
  if (!dyn || (flags & KF_QD0)) qdj = 0.f;
  if (!dyn || (flags & KF_QDD0)) qddj = 0.f;

  Xf X;
  joint_local<G == 64>(J, qj, X.R, X.p);  // past 32 joints as accurate as the thread-per-environment kernels
  if (!valid) X = identity_xf();
  T.prefix(X);
  const S6<float> col = valid ? jcol(J, X.R, X.p) : zero6<float>();
  const int u = J.vuser;
  // Streaming output stores (see st()), except up to 8 joints: their rows are
  // shorter than a 64-byte sector, and of plain stores the L2 cache merges the
  // pieces. 5-joint tree x 262144: 95 us streaming, 31 us so (42 with one
  // environment per 8 lanes, streaming); 8 joints x 65536 20.1 and 15.7, x 16384,
  // which the cache holds, 6.7 and 7.0.
  constexpr bool NT = G > 8;
  float *const prow = io.poses + row_at(env0, row, io.pose_env, L * 7);
  const int64_t pl = io.pose_link ? io.pose_link : 7;

  // Jacobian columns and link poses first: their stores drain while the
  // dynamics compute
  if ((flags & KF_JFULL) && live && valid) {
    float *Jb = io.J + env0 * 6 * nv + __umul24(row, 6 * nv) + u;
    st<NT>(col.l.x, Jb + 0 * nv); st<NT>(col.l.y, Jb + 1 * nv); st<NT>(col.l.z, Jb + 2 * nv);
    st<NT>(col.a.x, Jb + 3 * nv); st<NT>(col.a.y, Jb + 4 * nv); st<NT>(col.a.z, Jb + 5 * nv);
  }
  if ((flags & KF_POSES) && Mg->links_le1) {
    if (live && valid && J.link >= 0) {
      if (J.lident) {  // link frame = joint frame
        store_pose<NT>(prow + J.link * pl, X.R, X.p);
      } else {
        float Rw[9];
        mm(X.R, J.lR, Rw);
        store_pose<NT>(prow + J.link * pl, Rw, mv(X.R, load3(J.lp)) + X.p);
      }
    }
    if (live && g == 0 && Mg->root_link >= 0)
      store_pose_q<NT>(prow + Mg->root_link * pl, Mg->root_p, Mg->root_q);
  } else if (flags & KF_POSES) {
    for (int l0 = 0; l0 < L; l0 += T.S) {  // every lane takes part in the permutes
      const int l = l0 + g;
      const LinkRec<float> &LL = links_of(Mg)[l < L ? l : L - 1];
      const int jl = LL.joint < 0 ? 0 : LL.joint;
      const Xf W = bperm_xf(T.slot < io.pack.per_wave ? T.base4 + 4 * jl : 0, X);
      float Rw[9];
      mm(W.R, LL.R, Rw);
      V3<float> pw = mv(W.R, load3(LL.p)) + W.p;
      if (LL.joint < 0) {
#pragma unroll
        for (int k = 0; k < 9; ++k) Rw[k] = LL.R[k];
        pw = load3(LL.p);
      }
      if (live && l < L) store_pose<NT>(prow + l * pl, Rw, pw);
    }
  }
  // composite inertia of the subtree (additive form about the world origin),
  // summed with the RNEA forces when both are computed
  const bool do_crba = flags & KF_CRBA;
  float y[10];
  if (do_crba) {
    const AInertia<float> Ya = additive(world_inertia_fast(J, X.R, X.p));
    const float yv[10] = {Ya.m, Ya.h.x, Ya.h.y, Ya.h.z, Ya.I[0], Ya.I[1], Ya.I[2], Ya.I[3], Ya.I[4], Ya.I[5]};
#pragma unroll
    for (int i = 0; i < 10; ++i) y[i] = valid ? yv[i] : 0.f;
  }
  if (dyn) {
    S6<float> v = qdj * col;
    T.prefix(v);
    S6<float> a = qddj * col + qdj * crossm(v, col);
    T.prefix(a);
    if (!(flags & KF_NOGRAV)) a.l = a.l - V3<float>{Mg->gravity[0], Mg->gravity[1], Mg->gravity[2]};
    const WInertia<float> Y = world_inertia_fast(J, X.R, X.p);
    S6<float> f = valid ? inertia_apply(Y, a) + crossf(v, inertia_apply(Y, v)) : zero6<float>();
    if (do_crba) {
      // one subtree pass for the forces and the composite inertias
      float x[16] = {f.l.x, f.l.y, f.l.z, f.a.x, f.a.y, f.a.z};
#pragma unroll
      for (int i = 0; i < 10; ++i) x[6 + i] = y[i];
      T.template subtree<16>(x);
      f = {{x[0], x[1], x[2]}, {x[3], x[4], x[5]}};
#pragma unroll
      for (int i = 0; i < 10; ++i) y[i] = x[6 + i];
    } else {
      T.subtree(f);
    }
    if (live && valid) st<true>(dot6(col, f), io.tau + row_at(env0, row, io.ld_tau, nv) + u);
  }
  if (do_crba) {
    if (!dyn) T.template subtree<10>(y);
    AInertia<float> Yc;
    Yc.m = y[0];
    Yc.h = {y[1], y[2], y[3]};
#pragma unroll
    for (int i = 0; i < 6; ++i) Yc.I[i] = y[4 + i];
    const S6<float> Fj = apply(Yc, col);
    if (io.pack.dense) {
      // Deep trees: M is nearly full. Every lane publishes its column and force,
      // lane j reads those of all joints of its environment (one address across
      // it at a time) and stores row u of M, entry (i, u) for (u, i): at each i an
      // environment writes one contiguous row. A 32-joint chain x 65536: 109 us so,
      // 160 by the walk below; 30 joints 100 and 116; 16 joints 39 and 47.
      float4 *const cf = reinterpret_cast<float4 *>(lds);
      cf[T.lane * 3 + 0] = make_float4(col.l.x, col.l.y, col.l.z, col.a.x);
      cf[T.lane * 3 + 1] = make_float4(col.a.y, col.a.z, Fj.l.x, Fj.l.y);
      cf[T.lane * 3 + 2] = make_float4(Fj.l.z, Fj.a.x, Fj.a.y, Fj.a.z);
      wave_sync();
      const bool out = live && valid;
      const float4 *const ce = cf + (out ? T.base4 / 4 : 0) * 3;
      float *const Mcol = io.M + env0 * nv * nv + __umul24(row, nv * nv) + u;
#pragma unroll 4
      for (int i = 0; i < nj; ++i) {
        const float4 r0 = ce[i * 3 + 0], r1 = ce[i * 3 + 1], r2 = ce[i * 3 + 2];
        const S6<float> ci = {{r0.x, r0.y, r0.z}, {r0.w, r1.x, r1.y}};
        const S6<float> Fi = {{r1.z, r1.w, r2.x}, {r2.y, r2.z, r2.w}};
        // joint i's subtree size and user dof: on lane i, the first environment's
        const int sub_i = __builtin_amdgcn_readlane(T.size, i), ui = __builtin_amdgcn_readlane(u, i);
        const float dij = dot6(ci, Fj), dji = dot6(col, Fi);
        const bool i_anc_j = i <= g && g < i + sub_i, j_anc_i = g < i && i < g + T.size;
        if (out) Mcol[__umul24(ui, nv)] = i_anc_j ? dij : j_anc_i ? dji : 0.f;
      }
      return;
    }
    // M is nonzero between a joint and its ancestors: every lane publishes its
    // column, lane j walks its ancestors i and puts col_i . F_j at (i, j) and
    // (j, i) of the wavefront's LDS tile, whose environments then leave as one
    // contiguous run. 4095 environments of a 30-joint tree: 12.8 us with every lane
    // reading all 30 columns and forces and storing M row by row, 10.8 us so.
    AncestorRows<1> rows(lds);
    float *const tile = lds + AncestorRows<1>::kFloats;
    rows.put(T.lane, col, u, J.parent);
    zero_tile(tile, left * nv * nv, T.lane);
    wave_sync();
    float *const mine = tile + __umul24(T.slot, nv * nv);
    rows.template walk<G>(T, J, valid && live, io.pack.max_depth, [&](const S6<float>(&ci)[1], int ui, bool on) {
      const float v = dot6(ci[0], Fj);
      if (on) {
        mine[__umul24(ui, nv) + u] = v;
        mine[__umul24(u, nv) + ui] = v;
      }
    });
    wave_sync();
    float *const dst = io.M + env0 * nv * nv;
    copy_run<false>(tile, dst, left * nv * nv, T.lane, ((uintptr_t)dst & 15) == 0);
  }
}

// Forward recomputation + reverse pass (formulas in kernels_adjoint.hip).
// Pose gradients need one user link per joint (links_le1).
template <int G>
__device__ __forceinline__ void tree_vjp_body(const ModelTable<float> *M, int64_t B, int64_t env, const float *q,
                                              const float *qd, const float *qdd, const float *gsrc,
                                              const VjpArgs<float> &A) {
  const int g = threadIdx.x & (G - 1);
  const bool live = env < B;
  const int64_t e = live ? env : B - 1;
  const int nj = M->nj, nv = M->nv, L = M->nlinks;
  const bool dyn = A.gtau || A.tau_star;
  const bool valid = g < nj;
  const JointRec<float> &J = joints_of(M)[valid ? g : nj - 1];
  Tree<G> T;
  T.g = g;
  T.base4 = ((threadIdx.x & 63) & ~(G - 1)) * 4;
#pragma unroll
  for (int k = 0; k < Tree<G>::K; ++k) T.anc[k] = valid ? J.anc[k] : -1;
  T.size = valid ? J.subtree : 0;

  const int64_t qi = e * nv + (g < nv ? g : nv - 1);
  const float qu = q[qi], qdu = qd[qi], qddu = qdd[qi], gu = gsrc[qi];
  V3<float> ptarget = {0.f, 0.f, 0.f};
  if (A.p_target) ptarget = {A.p_target[e * 3], A.p_target[e * 3 + 1], A.p_target[e * 3 + 2]};
  const int src = T.base4 + 4 * J.vuser;
  float qj = bperm(src, qu), qdj = bperm(src, qdu), qddj = bperm(src, qddu), gj = bperm(src, gu);
  if (!valid) qj = qdj = qddj = gj = 0.f;
  if (!dyn) qdj = qddj = gj = 0.f;

  float s, c;
  joint_sincos(qj, &s, &c);
  Xf X;
  joint_world(J, qj, s, c, static_cast<const float *>(nullptr), V3<float>{0, 0, 0}, true, X.R, X.p);
  if (!valid) X = identity_xf();
  T.prefix(X);
  const S6<float> col = valid ? jcol(J, X.R, X.p) : zero6<float>();
  const int u = J.vuser;

  float loss = 0.f;
  S6<float> FP = zero6<float>();
  if (valid && J.link >= 0) {
    const int l = J.link;
    float Rw[9];
    mm(X.R, J.lR, Rw);
    const V3<float> pw = mv(X.R, load3(J.lp)) + X.p;
    if (A.gposes) {
      float quat[4];
      quat_branchless(Rw, quat);
      const float *gp7 = A.gposes + (e * L + l) * 7;
      const V3<float> gp = {gp7[0], gp7[1], gp7[2]}, gq = {gp7[4], gp7[5], gp7[6]};
      const V3<float> uq = {quat[1], quat[2], quat[3]};
      FP = {gp, cross(pw, gp) + 0.5f * (quat[0] * gq - gp7[3] * uq + cross(uq, gq))};
    } else if (A.p_target && l == A.ee_link) {
      const V3<float> d = pw - ptarget;
      loss += dot(d, d);
      const V3<float> gp = 2.f * d;
      FP = {gp, cross(pw, gp)};
    }
  }
  S6<float> Hw = zero6<float>(), QS = zero6<float>(), v = zero6<float>(), a = zero6<float>(), F = zero6<float>(),
            w = zero6<float>();
  if (dyn) {
    v = qdj * col;
    T.prefix(v);
    a = qddj * col + qdj * crossm(v, col);
    T.prefix(a);
    a.l = a.l - V3<float>{M->gravity[0], M->gravity[1], M->gravity[2]};
    const WInertia<float> Y = world_inertia_fast(J, X.R, X.p);
    F = valid ? inertia_apply(Y, a) + crossf(v, inertia_apply(Y, v)) : zero6<float>();
    T.subtree(F);
    const float tj = dot6(col, F);
    if (A.tau && live && valid) A.tau[e * nv + u] = tj;
    if (A.tau_star) {
      const float d = valid ? tj - gj : 0.f;
      loss += d * d;
      gj = 2.f * d;
    }
    w = gj * col;
    T.prefix(w);
    const S6<float> Iw = inertia_apply(Y, w), Iv = inertia_apply(Y, v);
    if (valid) {
      Hw = Iw;
      QS = crossf(w, Iv) - crossf(v, Iw) + inertia_apply(Y, crossm(v, w));
    }
  }
  float acc[18] = {Hw.l.x, Hw.l.y, Hw.l.z, Hw.a.x, Hw.a.y, Hw.a.z, QS.l.x, QS.l.y, QS.l.z,
                   QS.a.x, QS.a.y, QS.a.z, FP.l.x, FP.l.y, FP.l.z, FP.a.x, FP.a.y, FP.a.z};
  T.template subtree<18>(acc);
  Hw = {{acc[0], acc[1], acc[2]}, {acc[3], acc[4], acc[5]}};
  QS = {{acc[6], acc[7], acc[8]}, {acc[9], acc[10], acc[11]}};
  FP = {{acc[12], acc[13], acc[14]}, {acc[15], acc[16], acc[17]}};
  if (live && valid) {
    float dq = dot6(col, FP);
    if (dyn) {
      const S6<float> wl = w - gj * col, vl = v - qdj * col;
      const S6<float> al = a - qddj * col - qdj * crossm(v, col);
      dq += dot6(col, crossf(vl, QS + crossf(vl, Hw)) - crossf(wl, F) - crossf(al, Hw));
      if (A.dqd) A.dqd[e * nv + u] = -dot6(col, QS + 2.f * crossf(vl, Hw));
      if (A.dqdd) A.dqdd[e * nv + u] = dot6(col, Hw);
    }
    if (A.dq) A.dq[e * nv + u] = dq;
  }
  if ((A.tau_star || A.p_target) && A.loss) {
    loss = group_sum<G>(g, T.base4, loss);
    if (live && g == 0) A.loss[e] = loss;
  }
}

__device__ __forceinline__ void stage_table(float4 *s_tab, const ModelTable<float> *Mg) {
  const int n4 = (int)((kHeaderBytes + sizeof(JointRec<float>) * Mg->nj) / 16);
  const float4 *src = reinterpret_cast<const float4 *>(Mg);
  for (int i = threadIdx.x; i < n4; i += blockDim.x) s_tab[i] = src[i];
}

template <int G, bool SPARE>
__global__ __launch_bounds__(64 * tree_waves(G)) void k_tree_fused(const ModelTable<float> *__restrict__ Mg, int64_t B,
                                                                   int flags, TreeIO io, int wave_floats) {
  __shared__ float4 s_tab[(kHeaderBytes + sizeof(JointRec<float>) * G) / 16];
  extern __shared__ __align__(16) float s_rows[];  // wave_floats per wavefront
  stage_table(s_tab, Mg);
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  tree_body<G, SPARE>(reinterpret_cast<const ModelTable<float> *>(s_tab), Mg, B, blockIdx.x * (int64_t)tree_waves(G) + w,
                      flags, io, s_rows + w * wave_floats);
}

template <int G>
__global__ __launch_bounds__(256) void k_tree_vjp(const ModelTable<float> *__restrict__ Mg, int64_t B,
                                                  const float *__restrict__ q, const float *__restrict__ qd,
                                                  const float *__restrict__ qdd, const float *__restrict__ gsrc,
                                                  VjpArgs<float> A) {
  __shared__ float4 s_tab[kTreeTableWords4];
  stage_table(s_tab, Mg);
  __syncthreads();
  const int64_t env = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / G;
  tree_vjp_body<G>(reinterpret_cast<const ModelTable<float> *>(s_tab), B, env, q, qd, qdd, gsrc, A);
}

// Link poses and velocities written into a GPU simulator's body-state rows
// (13 floats: p xyz | q wxyz | v xyz | w xyz, world frame). Row 0 of an
// environment holds user link 0 (the simulator's root link): its pose and
// velocity are read first and place the articulation. With (R_m, p_m) a link's
// pose and (w_m, v_m) its angular and origin velocity in the model frame
// (from q, qd), and (R_0, p_0, w_0) read from row 0:
//   R_b = R_0 R_m0^T, p_b = p_0 - R_b p_m0          (the model frame in the world)
//   w_b = w_0 - R_b w_m0, u_b = v_0 - R_b v_m0      (its motion; u_b at point p_0)
//   pose_l = (R_b R_ml, R_b p_ml + p_b),  w_l = w_b + R_b w_ml,
//   v_l = u_b + w_b x (p_l - p_0) + R_b v_ml + w_l x (R_l c_l),
// v_0 being row 0's origin velocity (its stored centre-of-mass velocity minus
// w_0 x R_0 c_0) and the last term moving each origin velocity to the link's
// centre of mass c_l. Without qd only the poses (first 7 floats) are written.
struct LinkStateIO {
  const float *q, *qd;
  int64_t ld_q, ld_qd;
  float *body;
  int64_t env_stride, link_stride;
};

// Model-frame pose and velocity (angular, at the link origin) of user link l
// from the group's joint transforms X and joint velocities v (every lane calls
// this with its own l: the permutes run in all lanes).
template <int G>
__device__ __forceinline__ void link_model_state(const Tree<G> &T, const LinkRec<float> &LL, const Xf &X,
                                                 const S6<float> &v, float *Rm, V3<float> &pm, V3<float> &wm,
                                                 V3<float> &vm) {
  const int jl = LL.joint < 0 ? 0 : LL.joint;
  const Xf W = bperm_xf(T.base4 + 4 * jl, X);
  const S6<float> Vj = bperm6(T.base4 + 4 * jl, v);
  mm(W.R, LL.R, Rm);
  pm = mv(W.R, load3(LL.p)) + W.p;
  wm = Vj.a;
  vm = Vj.l + cross(Vj.a, pm);
  if (LL.joint < 0) {  // on the universe: fixed in the model frame
#pragma unroll
    for (int k = 0; k < 9; ++k) Rm[k] = LL.R[k];
    pm = load3(LL.p);
    wm = vm = V3<float>{0.f, 0.f, 0.f};
  }
}

template <int G>
__global__ __launch_bounds__(256) void k_link_state(const ModelTable<float> *__restrict__ Mg, int64_t B,
                                                    LinkStateIO io) {
  __shared__ float4 s_tab[kTreeTableWords4];
  stage_table(s_tab, Mg);
  __syncthreads();
  const ModelTable<float> *M = reinterpret_cast<const ModelTable<float> *>(s_tab);
  const int64_t env = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / G;
  const int g = threadIdx.x & (G - 1);
  const bool live = env < B;
  const int64_t e = live ? env : B - 1;
  const int nj = M->nj, nv = M->nv, L = M->nlinks;
  const bool vel = io.qd != nullptr;
  const bool valid = g < nj;
  const JointRec<float> &J = joints_of(M)[valid ? g : nj - 1];
  Tree<G> T;
  T.g = g;
  T.base4 = ((threadIdx.x & 63) & ~(G - 1)) * 4;
#pragma unroll
  for (int k = 0; k < Tree<G>::K; ++k) T.anc[k] = valid ? J.anc[k] : -1;
  T.size = valid ? J.subtree : 0;

  const int gc = g < nv ? g : nv - 1;
  const float qu = io.q[e * io.ld_q + gc], qdu = vel ? io.qd[e * io.ld_qd + gc] : 0.f;
  const int src = T.base4 + 4 * J.vuser;
  float qj = bperm(src, qu), qdj = bperm(src, qdu);
  if (!valid) qj = qdj = 0.f;
  float s, c;
  joint_sincos(qj, &s, &c);
  Xf X;
  joint_world(J, qj, s, c, static_cast<const float *>(nullptr), V3<float>{0, 0, 0}, true, X.R, X.p);
  if (!valid) X = identity_xf();
  T.prefix(X);
  S6<float> v = zero6<float>();
  if (vel) {
    v = valid ? qdj * jcol(J, X.R, X.p) : zero6<float>();
    T.prefix(v);  // spatial velocity of each joint body, model frame, linear part at the model origin
  }

  // row 0: user link 0's world pose and velocity (read before any row is written)
  float *row = io.body + e * io.env_stride;
  const V3<float> p0 = {row[0], row[1], row[2]};
  float qw = row[3], qx = row[4], qy = row[5], qz = row[6];
  const float rn = rsqrtf(qw * qw + qx * qx + qy * qy + qz * qz);
  qw *= rn; qx *= rn; qy *= rn; qz *= rn;
  const float R0[9] = {1.f - 2.f * (qy * qy + qz * qz), 2.f * (qx * qy - qw * qz), 2.f * (qx * qz + qw * qy),
                       2.f * (qx * qy + qw * qz), 1.f - 2.f * (qx * qx + qz * qz), 2.f * (qy * qz - qw * qx),
                       2.f * (qx * qz - qw * qy), 2.f * (qy * qz + qw * qx), 1.f - 2.f * (qx * qx + qy * qy)};
  V3<float> vc0 = {0.f, 0.f, 0.f}, w0 = {0.f, 0.f, 0.f};
  if (vel) {
    vc0 = {row[7], row[8], row[9]};
    w0 = {row[10], row[11], row[12]};
  }
  const LinkRec<float> &L0 = links_of(Mg)[0];
  float Rm0[9];
  V3<float> pm0, wm0, vm0;
  link_model_state<G>(T, L0, X, v, Rm0, pm0, wm0, vm0);
  float Rb[9];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int k = 0; k < 3; ++k)
      Rb[3 * i + k] = R0[3 * i] * Rm0[3 * k] + R0[3 * i + 1] * Rm0[3 * k + 1] + R0[3 * i + 2] * Rm0[3 * k + 2];
  const V3<float> pb = p0 - mv(Rb, pm0);
  const V3<float> wb = w0 - mv(Rb, wm0);
  const V3<float> ub = vc0 - cross(w0, mv(R0, load3(L0.c))) - mv(Rb, vm0);

  for (int l0 = 0; l0 < L; l0 += G) {  // every lane takes part in the permutes
    const int l = l0 + g;
    const LinkRec<float> &LL = links_of(Mg)[l < L ? l : L - 1];
    float Rm[9];
    V3<float> pm, wm, vm;
    link_model_state<G>(T, LL, X, v, Rm, pm, wm, vm);
    float Rw[9];
    mm(Rb, Rm, Rw);
    const V3<float> pw = mv(Rb, pm) + pb;
    if (live && l < L) {
      float *out = row + l * io.link_stride;
      store_pose(out, Rw, pw);
      if (vel) {
        const V3<float> ww = wb + mv(Rb, wm);
        const V3<float> vc = ub + cross(wb, pw - p0) + mv(Rb, vm) + cross(ww, mv(Rw, load3(LL.c)));
        out[7] = vc.x; out[8] = vc.y; out[9] = vc.z;
        out[10] = ww.x; out[11] = ww.y; out[12] = ww.z;
      }
    }
  }
}

// Heterogeneous launch: block ranges map to segments (one tree type each).
__global__ __launch_bounds__(256) void k_hetero(HeteroArgs args, int flags, int wave_floats) {
  __shared__ float4 s_tab[kTreeTableWords4];
  extern __shared__ __align__(16) float s_rows[];  // wave_floats per wavefront
  int s = 0;
  while (s + 1 < args.nseg && (int64_t)blockIdx.x >= args.seg[s + 1].block0) ++s;
  const HeteroSegment &S = args.seg[s];
  stage_table(s_tab, S.tab);
  __syncthreads();
  const ModelTable<float> *M = reinterpret_cast<const ModelTable<float> *>(s_tab);
  const TreeIO io{S.q, S.qd ? S.qd : S.q, S.qdd ? S.qdd : S.q, S.poses, S.J, S.tau, S.M, S.pack};
  int f = flags;
  if (!S.poses) f &= ~KF_POSES;
  if (!S.J) f &= ~KF_JFULL;
  if (!S.tau) f &= ~KF_RNEA;
  if (!S.M) f &= ~KF_CRBA;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t wave = ((int64_t)blockIdx.x - S.block0) * 4 + w;
  float *const lds = s_rows + w * wave_floats;
  switch (S.pack.width + (S.pack.spare ? 1 : 0)) {  // uniform per block
    case 8: tree_body<8, false>(M, S.tab, S.B, wave, f, io, lds); break;
    case 9: tree_body<8, true>(M, S.tab, S.B, wave, f, io, lds); break;
    case 16: tree_body<16, false>(M, S.tab, S.B, wave, f, io, lds); break;
    case 17: tree_body<16, true>(M, S.tab, S.B, wave, f, io, lds); break;
    case 32: tree_body<32, false>(M, S.tab, S.B, wave, f, io, lds); break;
    default: tree_body<32, true>(M, S.tab, S.B, wave, f, io, lds); break;
  }
}

}  // namespace

int tree_group(int nj) { return nj < 1 ? 0 : nj <= 8 ? 8 : nj <= 16 ? 16 : nj <= 32 ? 32 : 0; }

// lanes = 0, the default, is back to back at every batch. Fused kinematics, us a
// launch, packed / smallest group that holds the joints (environments a
// wavefront):
//   batch             1024        4096        8192        16384       65536       262144
//   9 joints (7/4)    5.5/5.2     5.8/5.5     6.5/6.3     8.4/8.7    26.6/25.6   69.5/94.7
//   18 joints (3/2)   6.1/6.1     7.4/7.3     9.0/10.6   14.9/18.0   44.7/60.8    167/235
//   30 joints (2/2)   6.4/6.3     7.7/7.6    11.1/10.9   19.1/18.7   64.9/64.2    251/246
// Below about 8192 environments, where fewer wavefronts have more to do each, the
// groups are up to 5 % faster; the mixed launch of four trees x 8192 takes 12.9
// packed and 12.3 with 8 / 16 / packed / 32, which the autotuner finds.
TreePacking tree_packing(int nj, int nlinks, int max_depth, int lanes) {
  TreePacking p;
  p.nj = nj;
  p.nlinks = nlinks;
  p.max_depth = max_depth;
  p.rounds = 0;
  while ((1 << p.rounds) < max_depth) ++p.rounds;
  // M row by row where a joint has most others as ancestors; past 32 joints the
  // walk over the ancestors is the faster one at small batches (64 joints x 64:
  // 13.7 us, 15.5 row by row).
  p.dense = nj <= 32 && 4 * max_depth > 3 * nj;
  p.stride = lanes ? lanes : nj;
  p.per_wave = 64 / p.stride;
  p.magic = 65536 / p.stride + 1;
  p.spare = p.stride > nj || p.per_wave * p.stride < 64;
  const int n = nj + p.spare;
  p.width = n <= 8 ? 8 : n <= 16 ? 16 : n <= 32 ? 32 : 64;
  return p;
}

namespace {
template <int G, bool SPARE>
void launch_fused(const ModelTable<float> *tab, dim3 grid, int64_t B, int flags, const TreeIO &io, hipStream_t s,
                   hipEvent_t ev0, hipEvent_t ev1) {
  constexpr int waves = tree_waves(G);
  const int floats = (flags & KF_CRBA) ? tree_wave_floats(io.pack) : 0;
  const unsigned lds = (unsigned)(waves * floats * (int)sizeof(float));
  if (ev0 || ev1)  // the kernel's own start and stop recorded into the caller's events
    hipExtLaunchKernelGGL((k_tree_fused<G, SPARE>), grid, dim3(64 * waves), lds, s, ev0, ev1, 0, tab, B, flags, io,
                          floats);
  else
    hipLaunchKernelGGL((k_tree_fused<G, SPARE>), grid, dim3(64 * waves), lds, s, tab, B, flags, io, floats);
}
}  // namespace

hipError_t launch_tree_fused(const ModelTable<float> *tab, int nj, int nlinks, int max_depth, int64_t B, int flags, const float *q,
                             const float *qd, const float *qdd, const KinOut<float> &out, hipStream_t s, int lanes,
                             hipEvent_t ev0, hipEvent_t ev1) {
  if (B <= 0) return hipSuccess;
  if (nj < 1 || nj > 64) return hipErrorNotSupported;
  if (lanes != 0 && ((lanes != 8 && lanes != 16 && lanes != 32) || lanes < nj)) return hipErrorInvalidValue;
  const bool use_qd = (flags & KF_RNEA) && !(flags & KF_QD0) && qd, use_qdd = (flags & KF_RNEA) && !(flags & KF_QDD0) && qdd;
  TreeIO io{q, use_qd ? qd : q, use_qdd ? qdd : q, out.poses, out.jfull, out.tau, out.M};
  io.pack = tree_packing(nj, nlinks, max_depth, lanes);
  io.ld_q = out.ld_q;
  io.ld_qd = use_qd ? out.ld_qd : out.ld_q;
  io.ld_qdd = use_qdd ? out.ld_qdd : out.ld_q;
  io.ld_tau = out.ld_tau;
  io.pose_env = out.pose_env;
  io.pose_link = out.pose_link;
  const int64_t per_block = tree_waves(io.pack.width) * io.pack.per_wave;
  const dim3 grid((unsigned)((B + per_block - 1) / per_block));
  if (!out.M) flags &= ~KF_CRBA;  // the CRBA rows are allocated only with an M output
  switch (io.pack.width + (io.pack.spare ? 1 : 0)) {
    case 8: launch_fused<8, false>(tab, grid, B, flags, io, s, ev0, ev1); break;
    case 9: launch_fused<8, true>(tab, grid, B, flags, io, s, ev0, ev1); break;
    case 16: launch_fused<16, false>(tab, grid, B, flags, io, s, ev0, ev1); break;
    case 17: launch_fused<16, true>(tab, grid, B, flags, io, s, ev0, ev1); break;
    case 32: launch_fused<32, false>(tab, grid, B, flags, io, s, ev0, ev1); break;
    case 33: launch_fused<32, true>(tab, grid, B, flags, io, s, ev0, ev1); break;
    case 64: launch_fused<64, false>(tab, grid, B, flags, io, s, ev0, ev1); break;
    default: launch_fused<64, true>(tab, grid, B, flags, io, s, ev0, ev1); break;
  }
  return hipGetLastError();
}

hipError_t launch_link_state(const ModelTable<float> *tab, int nj, int64_t B, const float *q, int64_t ld_q,
                             const float *qd, int64_t ld_qd, float *body, int64_t env_stride, int64_t link_stride,
                             hipStream_t s) {
  if (B <= 0) return hipSuccess;
  const int G = tree_group(nj);
  if (!G) return hipErrorNotSupported;
  LinkStateIO io{q, qd, ld_q, ld_qd, body, env_stride, link_stride};
  const int64_t per_block = 256 / G;
  dim3 grid((unsigned)((B + per_block - 1) / per_block));
  if (G == 8) hipLaunchKernelGGL(k_link_state<8>, grid, dim3(256), 0, s, tab, B, io);
  else if (G == 16) hipLaunchKernelGGL(k_link_state<16>, grid, dim3(256), 0, s, tab, B, io);
  else hipLaunchKernelGGL(k_link_state<32>, grid, dim3(256), 0, s, tab, B, io);
  return hipGetLastError();
}

hipError_t launch_tree_vjp(const ModelTable<float> *tab, int nj, int64_t B, const float *q, const float *qd,
                           const float *qdd, VjpArgs<float> a, hipStream_t s) {
  if (B <= 0) return hipSuccess;
  const int G = tree_group(nj);
  if (!G) return hipErrorNotSupported;
  const bool dyn = a.gtau || a.tau_star;
  if (!dyn) qd = qdd = q;
  const float *gsrc = a.tau_star ? a.tau_star : a.gtau ? a.gtau : q;
  const int64_t per_block = 256 / G;
  dim3 grid((unsigned)((B + per_block - 1) / per_block));
  if (G == 8) hipLaunchKernelGGL(k_tree_vjp<8>, grid, dim3(256), 0, s, tab, B, q, qd, qdd, gsrc, a);
  else if (G == 16) hipLaunchKernelGGL(k_tree_vjp<16>, grid, dim3(256), 0, s, tab, B, q, qd, qdd, gsrc, a);
  else hipLaunchKernelGGL(k_tree_vjp<32>, grid, dim3(256), 0, s, tab, B, q, qd, qdd, gsrc, a);
  return hipGetLastError();
}

hipError_t launch_hetero(HeteroArgs args, int flags, hipStream_t s) {
  int64_t blocks = 0;
  int floats = 0;
  for (int i = 0; i < args.nseg; ++i) {
    HeteroSegment &S = args.seg[i];
    if (!tree_group(S.nj) || (S.G != 0 && ((S.G != 8 && S.G != 16 && S.G != 32) || S.G < S.nj)))
      return hipErrorInvalidValue;
    S.pack = tree_packing(S.nj, S.nlinks, S.max_depth, S.G);
    S.block0 = blocks;
    blocks += (S.B + 4 * S.pack.per_wave - 1) / (4 * S.pack.per_wave);
    if (S.M && (flags & KF_CRBA)) floats = std::max(floats, tree_wave_floats(S.pack));
  }
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_hetero, dim3((unsigned)blocks), dim3(256), 4u * (unsigned)floats * (unsigned)sizeof(float), s,
                     args, flags, floats);
  return hipGetLastError();
}

}  // namespace sapamd
