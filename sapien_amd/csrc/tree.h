// Tree scans for the lanes-per-joint kernels: one environment per group of G
// lanes (G = 8, 16, 32 or 64), lane j owning joint j of the depth-first joint
// order. Root-to-joint prefixes by pointer jumping over the 2^k-th ancestors;
// subtree sums from doubling block sums over the preorder lane ranges.
#pragma once
#include <hip/hip_runtime.h>

#include "lanes.h"
#include "launch.h"
#include "spatial.h"

namespace sapamd {
namespace lanes {

template <class T> __device__ __forceinline__ S6<T> bperm6(int src4, S6<T> x) {
  return {{bperm(src4, x.l.x), bperm(src4, x.l.y), bperm(src4, x.l.z)},
          {bperm(src4, x.a.x), bperm(src4, x.a.y), bperm(src4, x.a.z)}};
}
template <class T> __device__ __forceinline__ XfT<T> bperm_xf(int src4, const XfT<T> &x) {
  XfT<T> o;
#pragma unroll
  for (int k = 0; k < 9; ++k) o.R[k] = bperm(src4, x.R[k]);
  o.p = {bperm(src4, x.p.x), bperm(src4, x.p.y), bperm(src4, x.p.z)};
  return o;
}

// Pointer jumping toward the root, at most log2(G) rounds; T is the scalar type
// of the scanned values. In FP64 the additions of a round sit in a branch (the
// exchanges do not: every lane has to take part), a mask per round where selects
// cost two instructions per value: a tree of 18 joints steps in 10.0 us instead
// of 10.4. In FP32 the selects are the faster form (a 9-joint arm 5.0 and 5.3 us).
template <int G, class T = float> struct Tree {
  static constexpr int K = G == 8 ? 3 : G == 16 ? 4 : G == 32 ? 5 : 6;
  int base4;
  int anc[K];
  int size;
  int g;
  static constexpr bool kLimit = G > 8;  // with few lanes a round costs less than asking whether it is needed
  int rounds = K;    // rounds the deepest joint needs (the same in every lane)
  bool full = true;  // a subtree may fill the group
  __device__ __forceinline__ void prefix(XfT<T> &x) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (kLimit && k >= rounds) break;
      const int a = anc[k];
      const XfT<T> y = bperm_xf(base4 + 4 * (a < 0 ? 0 : a), x);
      x = a >= 0 ? compose(y, x) : x;
    }
  }
  __device__ __forceinline__ void prefix(S6<T> &x) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int a = anc[k];
      if (kLimit && k >= rounds) break;
      const S6<T> y = bperm6(base4 + 4 * (a < 0 ? 0 : a), x);
      if constexpr (kBranch) {
        if (a >= 0) x = x + y;
      } else {
        x = sel(a >= 0, x + y, x);
      }
    }
  }
  static constexpr bool kBranch = sizeof(T) == 8;
  template <int N> static __device__ __forceinline__ void add_where(bool where, T (&x)[N], const T (&y)[N]) {
    if constexpr (kBranch) {
      if (where)
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] += y[i];
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = where ? x[i] + y[i] : x[i];
    }
  }
  // value of lane g + 2^k: a DPP row shift when the group lies in one 16-lane
  // row (G <= 16; the caller masks lanes whose source is past the group),
  // ds_bpermute otherwise
  template <int k> __device__ __forceinline__ T from_lane_above(T v) const {
    if constexpr (G <= 16) {
      return from_above<(1 << k)>(v);
    } else {
      const int src = g + (1 << k);
      return bperm(base4 + 4 * (src < G ? src : 0), v);
    }
  }
  // subtree sum of x over [g, g + size) (x = 0 on lanes without a joint)
  template <int N> __device__ __forceinline__ void subtree(T (&x)[N]) const {
    T blk[K][N];
    T cur[N];
#pragma unroll
    for (int i = 0; i < N; ++i) cur[i] = x[i];
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
      for (int i = 0; i < N; ++i) blk[k][i] = cur[i];
      if (kLimit && k == K - 1 && !full) break;  // the whole group's sum
      const bool in = g + (1 << k) < G;
      T y[N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        switch (k) {  // k is a constant once the loop is unrolled
          case 0: y[i] = from_lane_above<0>(cur[i]); break;
          case 1: y[i] = from_lane_above<1>(cur[i]); break;
          case 2: y[i] = from_lane_above<2>(cur[i]); break;
          case 3: y[i] = from_lane_above<3>(cur[i]); break;
          case 4: y[i] = from_lane_above<4>(cur[i]); break;
          default: y[i] = from_lane_above<5>(cur[i]); break;
        }
      }
      add_where(in, cur, y);
    }
    // blocks of size 2^K cover the whole group: size <= G
    T acc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = T(0);
    // every lane runs the query (ds_bpermute must not sit in divergent code);
    // size == G (a single-root tree filling the group) has no bits below K and
    // takes the full block instead
    int pos = g;
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
      const bool take = (size >> k) & 1;
      const int s4 = base4 + 4 * (pos < G ? pos : 0);
      T y[N];
#pragma unroll
      for (int i = 0; i < N; ++i) y[i] = bperm(s4, blk[k][i]);
      add_where(take, acc, y);
      pos += take ? (1 << k) : 0;
    }
    if ((!kLimit || full) && size >= G)
#pragma unroll
      for (int i = 0; i < N; ++i) acc[i] = cur[i];
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = acc[i];
  }
  __device__ __forceinline__ void subtree(S6<T> &f) const {
    T x[6] = {f.l.x, f.l.y, f.l.z, f.a.x, f.a.y, f.a.z};
    subtree<6>(x);
    f = {{x[0], x[1], x[2]}, {x[3], x[4], x[5]}};
  }
};

// The same scans over environments packed at a stride of S lanes (S >= nj, at
// most G), 64 / S of them per wavefront: any stride works because every exchange
// is a permute. SPARE: the wavefront has a lane without a joint (its values are
// the scans' neutral elements: identity, zero), which stands in for every
// missing source, so most selects go away; without it (no lane left over) the
// selects stay. Values and summation order are those of Tree<G>, bit for bit.
template <int G, bool SPARE> struct PackedTree {
  static constexpr int K = G == 8 ? 3 : G == 16 ? 4 : G == 32 ? 5 : 6;
  // With no lane to spare an environment of up to 16 lanes lies in one 16-lane
  // row (its stride divides 16): DPP row shifts in the sums. 16-joint tree x 16384,
  // M: 13.4 us so, 14.1 with permutes.
  static constexpr bool kInRows = !SPARE && G <= 16;
  int lane, slot, g;  // wave lane, environment within the wavefront, joint
  int S;
  int base4;          // 4 * the environment's first lane
  int spare4;         // 4 * the spare lane (SPARE)
  int rounds;         // pointer-jumping rounds the deepest joint needs
  int anc4[K];        // 4 * the lane of the 2^k-th ancestor (the spare lane past the root)
  uint32_t has;       // bit k: that ancestor exists
  int size;           // joints in the subtree, 0 without a joint

  __device__ __forceinline__ void place(const TreePacking &P) {
    lane = threadIdx.x & 63;
    S = P.stride;
    rounds = P.rounds;
    slot = __umul24(lane, P.magic) >> 16;
    const int first = __umul24(slot, S);
    g = lane - first;
    base4 = first * 4;
    spare4 = 4 * (S > P.nj ? P.nj : P.per_wave * S);
  }
  __device__ __forceinline__ void bind(const JointRec<float> &J, bool valid) {
    has = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int a = valid ? J.anc[k] : -1;
      anc4[k] = a >= 0 ? base4 + 4 * a : SPARE ? spare4 : base4;
      has |= a >= 0 ? 1u << k : 0u;
    }
    size = valid ? J.subtree : 0;
  }
  __device__ __forceinline__ void prefix(Xf &x) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) break;  // uniform; a round without ancestors changes nothing
      const Xf y = bperm_xf(anc4[k], x);
      const Xf z = compose(y, x);
      const bool in = (has >> k) & 1;
      if constexpr (SPARE) {  // identity times x is x
#pragma unroll
        for (int i = 0; i < 9; ++i) x.R[i] = z.R[i];
        x.p = {in ? z.p.x : x.p.x, in ? z.p.y : x.p.y, in ? z.p.z : x.p.z};  // an infinite p stays as it is
      } else {
        x = sel_xf(in, z, x);
      }
    }
  }
  __device__ __forceinline__ void prefix(S6<float> &x) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (k >= rounds) break;
      const S6<float> y = bperm6(anc4[k], x);
      if constexpr (SPARE) x = x + y;
      else x = sel((has >> k) & 1, x + y, x);
    }
  }
  // subtree sum of x over [g, g + size) (x = 0 on lanes without a joint)
  template <int N> __device__ __forceinline__ void subtree(float (&x)[N]) const {
    float blk[K][N], cur[N];
#pragma unroll
    for (int i = 0; i < N; ++i) cur[i] = x[i];
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
      for (int i = 0; i < N; ++i) blk[k][i] = cur[i];
      if (SPARE && k == K - 1) break;  // with a lane to spare no subtree has 2^K joints
      const bool in = size > 0 && g + (1 << k) < S;
      const int s4 = in ? base4 + 4 * (g + (1 << k)) : SPARE ? spare4 : 4 * lane;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if (k < 2) {  // one or two wavefront shifts: the LDS pipe is the busy one
          const float y = k == 0 ? wave_next(cur[i]) : wave_next(wave_next(cur[i]));
          cur[i] = in ? cur[i] + y : cur[i];
          continue;
        }
        if constexpr (kInRows) {
          const float y = k == 2 ? from_above<4>(cur[i]) : from_above<8>(cur[i]);
          cur[i] = in ? cur[i] + y : cur[i];
          continue;
        }
        const float y = bperm(s4, cur[i]);
        if constexpr (SPARE) cur[i] = cur[i] + y;
        else cur[i] = in ? cur[i] + y : cur[i];
      }
    }
    float acc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = 0.f;
    int pos = g;
#pragma unroll
    for (int k = K - 1; k >= 0; --k) {
      const bool take = (size >> k) & 1;
      const int s4 = take ? base4 + 4 * pos : SPARE ? spare4 : 4 * lane;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float y = bperm(s4, blk[k][i]);
        if constexpr (SPARE) acc[i] = acc[i] + y;
        else acc[i] = take ? acc[i] + y : acc[i];
      }
      pos += take ? (1 << k) : 0;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = !SPARE && size >= (1 << K) ? cur[i] : acc[i];
  }
  __device__ __forceinline__ void subtree(S6<float> &f) const {
    float x[6] = {f.l.x, f.l.y, f.l.z, f.a.x, f.a.y, f.a.z};
    subtree<6>(x);
    f = {{x[0], x[1], x[2]}, {x[3], x[4], x[5]}};
  }
};

// N world columns per joint in the wavefront's LDS with the joint's user dof and
// parent, for lanes that walk their joint's ancestors: matrices that are nonzero
// between a joint and its ancestors take max_depth steps a lane instead of nj.
template <int N> struct AncestorRows {
  static constexpr int kWords = 2 + 6 * N, kStride = (kWords + 3) & ~3;  // per lane, 16-byte aligned
  static constexpr int kFloats = 64 * kStride;
  float *buf;
  __device__ __forceinline__ explicit AncestorRows(float *lds) : buf(lds) {}
  __device__ __forceinline__ void put(int lane, const S6<float> &x, int u, int parent) { put(lane, &x, u, parent); }
  __device__ __forceinline__ void put(int lane, const S6<float> *x, int u, int parent) {
    float4 *r = reinterpret_cast<float4 *>(buf + lane * kStride);
    float w[kStride] = {};
#pragma unroll
    for (int n = 0; n < N; ++n) {
      w[6 * n + 0] = x[n].l.x; w[6 * n + 1] = x[n].l.y; w[6 * n + 2] = x[n].l.z;
      w[6 * n + 3] = x[n].a.x; w[6 * n + 4] = x[n].a.y; w[6 * n + 5] = x[n].a.z;
    }
    w[6 * N] = __builtin_bit_cast(float, u);
    w[6 * N + 1] = __builtin_bit_cast(float, parent);
#pragma unroll
    for (int i = 0; i < kStride / 4; ++i) r[i] = make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
  }
  // f(columns, user dof, exists) for this lane's joint and then its ancestors;
  // past the root, joint 0's values and exists = false.
  template <int G, class TREE, class F>
  __device__ __forceinline__ void walk(const TREE &T, const JointRec<float> &J, bool valid, int max_depth, F &&f) const {
    const float *first = buf + (valid ? T.base4 / 4 : 0) * kStride;
    int i = valid ? T.g : -1;
    uint32_t mask = valid ? J.ancmask : 0u;  // joints 0 .. 31
#pragma unroll 2
    for (int d = 0; d < max_depth; ++d) {
      if constexpr (G <= 32) {  // from the root: the reads of several steps can be in flight
        i = mask ? __builtin_ctz(mask) : -1;
        mask &= mask - 1u;
      }
      const float4 *r = reinterpret_cast<const float4 *>(first + (i < 0 ? 0 : i) * kStride);
      float w[kStride];
#pragma unroll
      for (int k = 0; k < kStride / 4; ++k) {
        const float4 q = r[k];
        w[4 * k] = q.x; w[4 * k + 1] = q.y; w[4 * k + 2] = q.z; w[4 * k + 3] = q.w;
      }
      S6<float> x[N];
#pragma unroll
      for (int n = 0; n < N; ++n)
        x[n] = {{w[6 * n], w[6 * n + 1], w[6 * n + 2]}, {w[6 * n + 3], w[6 * n + 4], w[6 * n + 5]}};
      f(x, __builtin_bit_cast(int, w[6 * N]), i >= 0);
      if constexpr (G > 32) i = i >= 0 ? __builtin_bit_cast(int, w[6 * N + 1]) : -1;
    }
  }
};

// The wavefront clears n floats (rounded up to 4) of its 16-byte aligned LDS.
__device__ __forceinline__ void zero_tile(float *tile, int n, int lane) {
  float4 *t4 = reinterpret_cast<float4 *>(tile);
  for (int i = lane; i < (n + 3) / 4; i += 64) t4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Sum over the G lanes of the group, result in lane 0.
template <int G> __device__ __forceinline__ float group_sum(int g, int base4, float x) {
#pragma unroll
  for (int d = 1; d < G; d *= 2) {
    const int src = g + d;
    const float y = bperm(base4 + 4 * (src < G ? src : 0), x);
    x = src < G ? x + y : x;
  }
  return x;
}

}  // namespace lanes
}  // namespace sapamd
