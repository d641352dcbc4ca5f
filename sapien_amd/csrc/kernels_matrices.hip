// Lanes-per-joint Coriolis matrices and per-link Jacobians (FP32) for trees of
// up to 64 joints, lane j owning joint j of the depth-first order, with the tree
// scans of tree.h: the Coriolis kernel packs environments back to back, a lane
// per joint, the Jacobian kernel gives each a group of 8, 16, 32 or 64 lanes.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lanes.h"
#include "launch.h"
#include "se3.h"
#include "spatial.h"
#include "tree.h"

namespace sapamd {

namespace {

using namespace lanes;

// Header and joint records of a G-lane model in LDS.
template <int G> constexpr int kTableWords = (int)((kHeaderBytes + sizeof(JointRec<float>) * G) / 16);

// Wavefronts per block: a wavefront's matrices take up to 20 KB of LDS.
constexpr int matrix_waves(int width) { return width > 32 ? 2 : 4; }

template <int G> __device__ __forceinline__ const ModelTable<float> *stage_joints(float4 *s_tab,
                                                                                 const ModelTable<float> *Mg) {
  const int n4 = (int)((kHeaderBytes + sizeof(JointRec<float>) * Mg->nj) / 16);
  const float4 *src = reinterpret_cast<const float4 *>(Mg);
  for (int i = threadIdx.x; i < n4; i += blockDim.x) s_tab[i] = src[i];
  __syncthreads();
  return reinterpret_cast<const ModelTable<float> *>(s_tab);
}

// World transform of this lane's joint from its angle (identity past the last
// joint). The library's sine and cosine: per-link Jacobians and C keep the
// accuracy they have in the thread-per-environment kernels.
template <int G>
__device__ __forceinline__ Xf joint_pose(const Tree<G> &T, const JointRec<float> &J, bool valid, float qj) {
  float s, c;
  sincosf(qj, &s, &c);
  Xf X;
  joint_world(J, qj, s, c, static_cast<const float *>(nullptr), V3<float>{0, 0, 0}, true, X.R, X.p);
  if (!valid) X = identity_xf();
  T.prefix(X);
  return X;
}

// C(q, qd) with the Christoffel-consistent per-body factorization of
// kernels_generic.hip, C = sum_i J_i^T (I_i Jdot_i + B_i J_i). About the world
// origin a body adds 10 inertia and 12 Coriolis numbers to its subtree sums
// (coriolis_terms in spatial.h) instead of two 6x6 matrices. With F1, G and H of
// each joint (coriolis_forces), C_kj = col_k . F1_j for k an ancestor-or-self of
// j and C_jk = G_j . dcol_k + H_j . col_k for a strict ancestor k: lane j walks its
// ancestors, and the wavefront's matrices are assembled in LDS and leave as one
// run. Environments are packed as in kernels_tree.hip.
//
// Bound: latency (a wavefront's chain of table copy, scans and walk takes about
// 7 us whatever the batch). 4095 environments of a 30-joint tree: 388 us in the
// thread-per-environment kernel (its two 6x6 matrices per joint live in scratch
// memory), 18.1 us with lane j reading all 30 joints' columns and storing its
// column of C row by row, 15.2 us here; the 14.7 MB of C take 3 us at a copy's
// rate.
template <int G, bool SPARE>
__global__ __launch_bounds__(64 * matrix_waves(G)) void k_tree_coriolis(const ModelTable<float> *__restrict__ Mg,
                                                                        int64_t B, const float *__restrict__ q,
                                                                        const float *__restrict__ qd,
                                                                        float *__restrict__ Cout, TreePacking pack,
                                                                        int wave_floats) {
  __shared__ float4 s_tab[kTableWords<G>];
  extern __shared__ __align__(16) float s_dyn[];  // wave_floats per wavefront
  const ModelTable<float> *M = stage_joints<G>(s_tab, Mg);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t env0 = (blockIdx.x * (int64_t)matrix_waves(G) + w) * pack.per_wave;
  if (env0 >= B) return;  // a wavefront of the last block
  const int left = (int)(B - env0 < pack.per_wave ? B - env0 : pack.per_wave);
  const int nj = pack.nj, nv = nj;
  PackedTree<G, SPARE> T;
  T.place(pack);
  const int g = T.g;
  const bool valid = T.slot < pack.per_wave && g < nj, live = T.slot < left;
  const JointRec<float> &J = joints_of(M)[valid ? g : nj - 1];
  T.bind(J, valid);
  const int at = __umul24(live ? T.slot : left - 1, nv) + (g < nv ? g : nv - 1);
  const float qu = q[env0 * nv + at], qdu = qd[env0 * nv + at];
  const int u = J.vuser, src = valid ? T.base4 + 4 * u : 0;
  float qj = bperm(src, qu), qdj = bperm(src, qdu);
  if (!valid) qj = qdj = 0.f;
  Xf X;
  joint_local<true>(J, qj, X.R, X.p);
  if (!valid) X = identity_xf();
  T.prefix(X);
  const S6<float> col = valid ? jcol(J, X.R, X.p) : zero6<float>();
  S6<float> v = qdj * col;
  T.prefix(v);
  const S6<float> dcol = crossm(v, col);

  float x[22];
  coriolis_terms(additive(world_inertia_fast(J, X.R, X.p)), v, x);
#pragma unroll
  for (int i = 0; i < 22; ++i) x[i] = valid ? x[i] : 0.f;
  T.template subtree<22>(x);
  S6<float> F1, Gc;
  V3<float> H;
  coriolis_forces(x, col, dcol, F1, Gc, H);

  AncestorRows<2> rows(s_dyn + w * wave_floats);
  float *const tile = rows.buf + AncestorRows<2>::kFloats;
  const S6<float> both[2] = {col, dcol};
  rows.put(T.lane, both, u, J.parent);
  zero_tile(tile, left * nv * nv, T.lane);
  wave_sync();
  float *const mine = tile + __umul24(T.slot, nv * nv);
  rows.template walk<G>(T, J, valid && live, pack.max_depth, [&](const S6<float>(&ci)[2], int ui, bool on) {
    const float down = dot6(Gc, ci[1]) + dot(H, ci[0].a), up = dot6(ci[0], F1);
    if (on) {
      mine[__umul24(u, nv) + ui] = down;
      mine[__umul24(ui, nv) + u] = up;  // the diagonal too: stored second
    }
  });
  wave_sync();
  float *const dst = Cout + env0 * nv * nv;
  copy_run<false>(tile, dst, left * nv * nv, T.lane, ((uintptr_t)dst & 15) == 0);
}

// Every link's Jacobian in the world and in the link frame, (B, L, 6, nv) each.
// A wavefront owns 64 / G consecutive environments, whose output rows are one
// contiguous run of links in memory. Once the joint transforms are known they
// and the Jacobian columns go to the wavefront's LDS, and the wavefront walks
// its run in chunks of whole links: the first lanes form the chunk's link
// poses, then every lane takes (link, dof) pairs and writes the 6 + 6 entries of
// a pair into two LDS tiles laid out as the output, and the tiles leave as
// contiguous stores. A tile holds one link of 64 dofs and up to kLinkChunk of a
// small robot; it takes the place of the joint records, so that four blocks
// share a CU's LDS. gridDim.y wavefronts split a run's chunks between them, each
// with its own forward kinematics, when the batch alone leaves the chip idle.
//
// Bound: output stores (2 x 24 nv bytes per link and environment) and, at small
// batches, the latency of a chunk's three passes. 1024 environments of a
// 40-joint chain (41 links, 80.6 MB): 1280 us in the thread-per-environment
// kernel, whose lanes write single floats a whole environment apart, 28.5 us
// with one wavefront per environment, 23.2 us with the run split three ways
// (17 us at a copy's rate); 64 environments 17.2 us split three ways, 8.2 us
// split to single chunks.
constexpr int kLinkTile = 512, kLinkChunk = 8;
struct LinkPose {
  float R[9], p[3];
  int joint, first;  // the link's joint (-1 = on the base), its environment's first lane
};

template <int G>
__global__ __launch_bounds__(256) void k_tree_link_jacobians(const ModelTable<float> *__restrict__ Mg, int64_t B,
                                                             const float *__restrict__ q, float *__restrict__ Jw,
                                                             float *__restrict__ Jl) {
  constexpr int kTile4 = 4 * 2 * kLinkTile / 4;
  __shared__ float4 s_tab[kTableWords<G> > kTile4 ? kTableWords<G> : kTile4];  // joint records, then the tiles
  __shared__ float s_col[4][6][64], s_X[4][12][64];
  __shared__ LinkPose s_link[4][kLinkChunk];
  __shared__ int s_joint[64], s_end[64];  // joint of each user dof; past the last joint of each joint's subtree
  const ModelTable<float> *M = stage_joints<G>(s_tab, Mg);
  const int nj = M->nj, nv = M->nv, L = M->nlinks;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  {
    const JointRec<float> *JR = joints_of(M);
    for (int j = threadIdx.x; j < nj; j += blockDim.x) {
      s_joint[JR[j].vuser] = j;
      s_end[j] = j + JR[j].subtree;
    }
    const int g = lane & (G - 1);
    const int64_t env = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / G;
    const int64_t e = env < B ? env : B - 1;
    const bool valid = g < nj;
    const JointRec<float> &J = JR[valid ? g : nj - 1];
    Tree<G> T;
    T.g = g;
    T.base4 = (lane & ~(G - 1)) * 4;
#pragma unroll
    for (int k = 0; k < Tree<G>::K; ++k) T.anc[k] = valid ? J.anc[k] : -1;
    const float qu = q[e * nv + (g < nv ? g : nv - 1)];
    float qj = bperm(T.base4 + 4 * J.vuser, qu);
    if (!valid) qj = 0.f;
    const Xf X = joint_pose<G>(T, J, valid, qj);
    const S6<float> col = jcol(J, X.R, X.p);
    const float cv[6] = {col.l.x, col.l.y, col.l.z, col.a.x, col.a.y, col.a.z};
#pragma unroll
    for (int r = 0; r < 6; ++r) s_col[wave][r][lane] = cv[r];
#pragma unroll
    for (int k = 0; k < 9; ++k) s_X[wave][k][lane] = X.R[k];
    s_X[wave][9][lane] = X.p.x;
    s_X[wave][10][lane] = X.p.y;
    s_X[wave][11][lane] = X.p.z;
  }
  __syncthreads();  // every wavefront is done with the joint records
  const int64_t env0 = (blockIdx.x * (int64_t)blockDim.x + (threadIdx.x & ~63)) / G;  // the wavefront's first
  if (env0 >= B) return;
  float *const tile = reinterpret_cast<float *>(s_tab) + wave * 2 * kLinkTile;
  const int run = (int)(B - env0 < 64 / G ? B - env0 : 64 / G) * L, width = 6 * nv;
  const int chunk = kLinkTile / width < kLinkChunk ? kLinkTile / width : kLinkChunk;
  for (int l0 = blockIdx.y * chunk; l0 < run; l0 += gridDim.y * chunk) {
    const int n = run - l0 < chunk ? run - l0 : chunk;
    if (lane < n) {
      const int first = (l0 + lane) / L * G;
      const LinkRec<float> &K = links_of(Mg)[(l0 + lane) % L];
      const int at = first + (K.joint < 0 ? 0 : K.joint);
      float R[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) R[k] = s_X[wave][k][at];
      const V3<float> p = {s_X[wave][9][at], s_X[wave][10][at], s_X[wave][11][at]};
      LinkPose P;
      mm(R, K.R, P.R);
      const V3<float> pw = mv(R, load3(K.p)) + p;
      P.p[0] = pw.x;
      P.p[1] = pw.y;
      P.p[2] = pw.z;
      P.joint = K.joint;
      P.first = first;
      s_link[wave][lane] = P;
    }
    wave_sync();
    for (int i = lane; i < n * nv; i += 64) {
      const int l = i / nv, u = i - l * nv;
      const LinkPose &P = s_link[wave][l];
      const int j = s_joint[u];
      S6<float> cw = zero6<float>(), cl = zero6<float>();
      if (j <= P.joint && P.joint < s_end[j]) {  // the joint carries the link
        const int at = P.first + j;
        cw = {{s_col[wave][0][at], s_col[wave][1][at], s_col[wave][2][at]},
              {s_col[wave][3][at], s_col[wave][4][at], s_col[wave][5][at]}};
        cl = to_local(P.R, load3(P.p), cw);
      }
      float *tw = tile + l * width + u, *tl = tw + kLinkTile;
      tw[0] = cw.l.x; tw[nv] = cw.l.y; tw[2 * nv] = cw.l.z;
      tw[3 * nv] = cw.a.x; tw[4 * nv] = cw.a.y; tw[5 * nv] = cw.a.z;
      tl[0] = cl.l.x; tl[nv] = cl.l.y; tl[2 * nv] = cl.l.z;
      tl[3 * nv] = cl.a.x; tl[4 * nv] = cl.a.y; tl[5 * nv] = cl.a.z;
    }
    wave_sync();
    const int64_t at = (env0 * L + l0) * width;
    float *const dst[2] = {Jw + at, Jl + at};
#pragma unroll
    for (int o = 0; o < 2; ++o)
      copy_run<true>(tile + o * kLinkTile, dst[o], n * width, lane, ((uintptr_t)dst[o] & 15) == 0);
    wave_sync();
  }
}

}  // namespace

int wave_group(int nj) { return nj < 1 || nj > 64 ? 0 : nj <= 8 ? 8 : nj <= 16 ? 16 : nj <= 32 ? 32 : 64; }

namespace {
template <int G, bool SPARE>
void launch_coriolis_packed(const ModelTable<float> *tab, int64_t B, const float *q, const float *qd, float *C,
                            const TreePacking &pack, hipStream_t s) {
  constexpr int waves = matrix_waves(G);
  const int floats = AncestorRows<2>::kFloats + ((pack.per_wave * pack.nj * pack.nj + 3) & ~3);
  const int64_t per_block = waves * pack.per_wave;
  hipLaunchKernelGGL((k_tree_coriolis<G, SPARE>), dim3((unsigned)((B + per_block - 1) / per_block)), dim3(64 * waves),
                     (unsigned)(waves * floats * (int)sizeof(float)), s, tab, B, q, qd, C, pack, floats);
}
}  // namespace

hipError_t launch_tree_coriolis(const ModelTable<float> *tab, int nj, int nlinks, int max_depth, int64_t B,
                                const float *q, const float *qd, float *C, hipStream_t s) {
  if (B <= 0) return hipSuccess;
  if (!wave_group(nj)) return hipErrorNotSupported;
  const TreePacking p = tree_packing(nj, nlinks, max_depth, 0);
  switch (p.width + (p.spare ? 1 : 0)) {
    case 8: launch_coriolis_packed<8, false>(tab, B, q, qd, C, p, s); break;
    case 9: launch_coriolis_packed<8, true>(tab, B, q, qd, C, p, s); break;
    case 16: launch_coriolis_packed<16, false>(tab, B, q, qd, C, p, s); break;
    case 17: launch_coriolis_packed<16, true>(tab, B, q, qd, C, p, s); break;
    case 32: launch_coriolis_packed<32, false>(tab, B, q, qd, C, p, s); break;
    case 33: launch_coriolis_packed<32, true>(tab, B, q, qd, C, p, s); break;
    case 64: launch_coriolis_packed<64, false>(tab, B, q, qd, C, p, s); break;
    default: launch_coriolis_packed<64, true>(tab, B, q, qd, C, p, s); break;
  }
  return hipGetLastError();
}

hipError_t launch_tree_link_jacobians(const ModelTable<float> *tab, int nj, int nlinks, int64_t B, const float *q,
                                      float *Jw, float *Jl, hipStream_t s) {
  if (B <= 0) return hipSuccess;
  const int G = wave_group(nj);
  if (!G) return hipErrorNotSupported;
  // as many wavefronts per run as give the chip about three blocks per CU;
  // past that a split only repeats the forward kinematics
  const int64_t blocks = (B * G + 255) / 256;
  const int chunk = std::min(kLinkChunk, kLinkTile / (6 * nj)), chunks = (64 / G * nlinks + chunk - 1) / chunk;
  const dim3 grid((unsigned)blocks, (unsigned)std::max<int64_t>(1, std::min<int64_t>(chunks, 768 / blocks)));
  switch (G) {
    case 8: hipLaunchKernelGGL(k_tree_link_jacobians<8>, grid, dim3(256), 0, s, tab, B, q, Jw, Jl); break;
    case 16: hipLaunchKernelGGL(k_tree_link_jacobians<16>, grid, dim3(256), 0, s, tab, B, q, Jw, Jl); break;
    case 32: hipLaunchKernelGGL(k_tree_link_jacobians<32>, grid, dim3(256), 0, s, tab, B, q, Jw, Jl); break;
    default: hipLaunchKernelGGL(k_tree_link_jacobians<64>, grid, dim3(256), 0, s, tab, B, q, Jw, Jl); break;
  }
  return hipGetLastError();
}

}  // namespace sapamd
