// Staged workgroups: C = 64 / H configurations shared by the W waves of a
// workgroup, with everything that depends only on the configuration computed
// once and kept in LDS.
//
//   1. every joint's local rotation (a lane per (configuration, joint)),
//   2. FK along the robot's paths, one wave per path: the poses of the
//      sphere-carrying and joint nodes,
//   3. the caller's work (sphere blocks, pairs, rows) split over all waves,
//      each reading the poses it needs.
//
// A lane-per-configuration walk of everything leaves a batch of B
// configurations B / 64 waves; here the walk that cannot be split (FK) runs
// once and the rest has W waves per C configurations.  H > 1 gives each
// configuration H lanes of a wave (lane = sub * C + configuration), which
// share the spheres of a block, so that a batch of a few thousand
// configurations still gives every CU a workgroup.
//
// All tables are laid out [index][configuration], so the lanes of a wave read
// consecutive words.  The arithmetic of a pose is that of run_fk (fk.hpp).
#pragma once

#include "device.hpp"

namespace pmp {

// Configurations (64 / H) and waves (W) of a workgroup for a batch of B: the
// fewest configurations while every CU then gets one workgroup at most, with
// 16 waves each; once a CU has several workgroups, 8 waves, and 4 when the
// robot has so few sphere blocks that most of 8 would wait for the walk.
// Measured (us), 7R arm, 32 primitives: evaluate of 4,096 configurations 19.1
// with H = 4, 24 with H = 1; of 8,192 22.0 with H = 2, 24.3 with H = 1; of
// 32,768 35 with 8 waves, 60 with 16; of 65,536 50 with 4 waves, 63 with 8.
// Validity of 1,000: 13.5 with H = 8, 14.1 with H = 4, 16.7 with H = 1; of
// 32,768 24 with 8 waves, 32 with 16; of 131,072 55 with 4 waves, 65 with 8.
// A robot whose tables take more than half of a CU's LDS has one workgroup there,
// which then gets 16 waves (100,000 configurations of 31 joints on a
// floating base: validity 350 us with 8, 207 with 16; evaluate 488 and 333; of 60
// joints 1,150 and 761, 1,297 and 842).
struct StageShape {
  int H, W;
};
inline StageShape stage_shape(int64_t B, int n_blocks) {
  StageShape s;
  s.H = B <= 8 * kCus ? 8 : (B <= 16 * kCus ? 4 : (B <= 32 * kCus ? 2 : 1));
  s.W = B <= 64 * kCus ? 16 : (B > 128 * kCus && n_blocks <= 8 ? 4 : 8);
  return s;
}

// The waves of a workgroup, at most W, with which a launch of n workgroups stays
// below the 2^32 threads a launch may have.
inline int waves_of_launch(int64_t n, int W) {
  while (W > 1 && n * 64 * W > 0xffffffffll) W /= 2;
  return W;
}

// Touches [p, p + bytes) through the scalar data cache, a line in n_parts: for
// waves that would otherwise wait while another one walks, so that the tables
// the whole workgroup is about to read are in the cache it shares.
__device__ __forceinline__ void warm_scalar(const void* p, int bytes, int part, int n_parts) {
  const int32_t* w = reinterpret_cast<const int32_t*>(p);
  for (int i = part * 16; i < bytes / 4; i += n_parts * 16) {
    const int v = cload(w, i);
    asm volatile("" ::"s"(v));
  }
}

template <int H>
struct Stage {
  static constexpr int C = 64 / H;           // configurations of the workgroup
  static constexpr int NK = kBlockSpheres / H;  // spheres of a block a lane takes
  float* lds;
  StageLds L;
  int lane, w, W, cfg, sub;
  __device__ __forceinline__ Stage(float* base, const StageLds& lay)
      : lds(base),
        L(lay),
        lane(threadIdx.x & 63),
        w(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))),
        W(blockDim.x >> 6),
        cfg(lane & (C - 1)),
        sub(H == 1 ? 0 : lane / C) {}

  // Every joint's local rotation (origin times joint), or its displacement in
  // word 0 of a prismatic one; and the path entries.
  template <class QS>
  __device__ __forceinline__ void joints(const KinArgs<float>& ka, const QS& qs, bool taylor) const {
    if (L.path >= 0)
      for (int i = threadIdx.x; i < 4 * ka.n_path_entries; i += blockDim.x)
        reinterpret_cast<float4*>(lds + L.path)[i] = reinterpret_cast<const float4*>(ka.path)[i];
    for (int i = w * H + sub; i < ka.n_joints; i += W * H) {
      const DevJoint jt = H == 1 ? cload(ka.joints, i) : ka.joints[i];
      const double v = qs.get(jt.q_col);
      Q4<float> lq{(float)v, 0.0f, 0.0f, 0.0f};
      if (jt.revolute) {
        const float x = (float)v * 0.5f;
        float s, c;
        if (taylor)
          taylor_sincos<float>(x, s, c);
        else
          exact_sincos(x, s, c);
        const Q4<float> jq{s * jt.axis[0], s * jt.axis[1], s * jt.axis[2], c};
        lq = jt.identity ? jq : qmul(Q4<float>{jt.quat[0], jt.quat[1], jt.quat[2], jt.quat[3]}, jq);
      }
      float* p = lds + L.joints + 4 * i * C + cfg;
      p[0] = lq.x;
      p[C] = lq.y;
      p[2 * C] = lq.z;
      p[3 * C] = lq.w;
    }
  }

  // The paths of this wave (path p goes to wave p mod W); joints() of every
  // wave must be complete.  A node costs its dependent chain (about 65 vector
  // instructions of one wave): the entries are read from LDS two ahead and the
  // joints' words one ahead.  (Entries read by scalar loads meet the LDS reads
  // in one wait counter, which then waits for both: 1,000 configurations of the
  // 14-joint robot 16.8 us, so 15.5; 512 motions of it 50.9 and 48.2.)
  struct Entry {
    float4 quat, trans_axis0, axis12_kind_identity, joint_pose;
  };
  __device__ __forceinline__ Entry entry(const KinArgs<float>& ka, int e) const {
    if (L.path >= 0) {
      const float4* p = reinterpret_cast<const float4*>(lds + L.path) + 4 * e;
      return {p[0], p[1], p[2], p[3]};
    }
    const float4* p = reinterpret_cast<const float4*>(ka.path + e);
    return {p[0], p[1], p[2], p[3]};
  }
  __device__ __forceinline__ Q4<float> joint_words(const Entry& e) const {
    const float* p = lds + L.joints + 4 * __float_as_int(e.joint_pose.x) * C + cfg;
    return {p[0], p[C], p[2 * C], p[3 * C]};
  }
  template <class QS>
  __device__ __forceinline__ void walk(const KinArgs<float>& ka, const QS& qs) const {
    for (int p = w; p < ka.n_paths; p += W) {
      Pose<float> P = base_pose(ka, qs);
      const int e_end = cload(ka.path_at, p + 1), e_begin = cload(ka.path_at, p);
      Entry cur = entry(ka, e_begin), next = entry(ka, min(e_begin + 1, e_end - 1));
      Q4<float> jq = joint_words(cur);
      for (int e = e_begin; e < e_end; ++e) {
        const Q4<float> jq_next = joint_words(next);
        const Entry after = entry(ka, min(e + 2, e_end - 1));
        const V3<float> lt{cur.trans_axis0.x, cur.trans_axis0.y, cur.trans_axis0.z};
        const Q4<float> oq{cur.quat.x, cur.quat.y, cur.quat.z, cur.quat.w};
        const int kind = __builtin_amdgcn_readfirstlane(__float_as_int(cur.axis12_kind_identity.z));
        const int pose = __builtin_amdgcn_readfirstlane(__float_as_int(cur.joint_pose.y));
        switch (kind) {
          case PMP_NODE_ROOT:
            break;
          case PMP_NODE_FIXED:
            P = compose(P, oq, lt,
                        __builtin_amdgcn_readfirstlane(__float_as_int(cur.axis12_kind_identity.w)) != 0);
            break;
          case PMP_NODE_REVOLUTE:
            P = compose(P, jq, lt, false);
            break;
          case PMP_NODE_PRISMATIC: {
            const float v = jq.x;
            const V3<float> t2{lt.x + cur.trans_axis0.w * v, lt.y + cur.axis12_kind_identity.x * v,
                               lt.z + cur.axis12_kind_identity.y * v};
            P = compose(P, oq, t2, true);
            break;
          }
          default: {  // PMP_NODE_TRANSLATION
            const M3<float> R = qmat(P.q);
            P.t = add(P.t, mv3(R, lt));
            break;
          }
        }
        if (pose >= 0) pose_set(pose, P);
        cur = next;
        next = after;
        jq = jq_next;
      }
    }
  }

  // With H > 1 the lanes of a configuration hold the same value and write it
  // to the same word.
  __device__ __forceinline__ void pose_set(int i, const Pose<float>& P) const {
    float* p = lds + L.poses + 7 * i * C + cfg;
    p[0] = P.q.x;
    p[C] = P.q.y;
    p[2 * C] = P.q.z;
    p[3 * C] = P.q.w;
    p[4 * C] = P.t.x;
    p[5 * C] = P.t.y;
    p[6 * C] = P.t.z;
  }
  // i may differ between lanes
  __device__ __forceinline__ Pose<float> pose(int i) const {
    const float* p = lds + L.poses + 7 * i * C + cfg;
    return {{p[0], p[C], p[2 * C], p[3 * C]}, {p[4 * C], p[5 * C], p[6 * C]}};
  }
  // World axis and origin of q column j (wave-uniform or not); false when the
  // column moves no sphere.
  template <class QS>
  __device__ __forceinline__ bool frame(const KinArgs<float>& ka, const QS& qs, int j, V3<float>& a,
                                        V3<float>& o) const {
    if (j >= ka.n_q_cols) {
      base_columns(ka, base_pose(ka, qs), qs, [&](int col, V3<float> ca, V3<float> co) {
        if (col == j) {
          a = ca;
          o = co;
        }
      });
      return true;
    }
    const DevColumn col = ka.columns[j];
    if (col.pose < 0) return false;
    const Pose<float> P = pose(col.pose);
    a = qrot(P.q, V3<float>{col.axis[0], col.axis[1], col.axis[2]});
    o = P.t;
    return true;
  }

  // f(column, its derivative at point c of node `node`) for every joint that
  // moves the node (robots whose q columns drive several joints).
  template <class F>
  __device__ __forceinline__ void joint_columns(const KinArgs<float>& ka, int node, V3<float> c, F&& f) const {
    for (int i = 0; i < ka.n_joints; ++i) {
      const DevJoint jt = cload(ka.joints, i);
      if (!moves_node(ka, jt.node, node)) continue;
      const Pose<float> P = pose(jt.pose);
      const V3<float> a = qrot(P.q, V3<float>{jt.axis[0], jt.axis[1], jt.axis[2]});
      f(jt.q_col, jt.revolute ? cross(a, pmp::sub(c, P.t)) : a);
    }
  }

  // The n (at most NK) spheres of block bk this lane takes: centres and radii.
  __device__ __forceinline__ void spheres(const KinArgs<float>& ka, int bi, const DevSphereBlock& bk,
                                          const Pose<float>& P, const M3<float>& R, V3<float> (&c)[NK],
                                          float (&r)[NK], int& n) const {
    n = H == 1 ? bk.n : bk.n - sub * NK;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      c[k] = P.t;
      r[k] = 0.0f;
      if constexpr (H == 1) {
        if (k < n) {
          c[k] = add(mv3(R, V3<float>{bk.s[k][0], bk.s[k][1], bk.s[k][2]}), P.t);
          r[k] = bk.s[k][3];
        }
      } else if (k < n) {
        const Quad4 s = reinterpret_cast<const Quad4*>(ka.blocks[bi].s)[sub * NK + k];  // a sphere a lane
        c[k] = add(mv3(R, V3<float>{s.v[0], s.v[1], s.v[2]}), P.t);
        r[k] = s.v[3];
      }
    }
  }
};

}  // namespace pmp
