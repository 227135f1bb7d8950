// Device functions shared by the kernels: wave reductions, box distances, the
// walk over a point cloud's tiles for a block of spheres, and the base columns.
#pragma once

#include <float.h>
#include <limits.h>

#include "fk.hpp"
#include "launch.h"

namespace pmp {

constexpr float kCutoff = 0.1f;  // SphereCollisionCst::cutoff_dist_ (primitive_sphere_collision.hpp:115)
template <class T>
__device__ __forceinline__ DevPrim<T> prim_at(const SceneArgs<T>& sc, int p) {
  return cload(reinterpret_cast<const DevPrim<T>*>(sc.prims), p);
}

// Whether node a is n or above it (robots with ka.shared).
__device__ __forceinline__ bool moves_node(const KinArgs<float>& ka, int a, int n) {
  return (ka.above[n * kNodeWords + (a >> 5)] >> (a & 31)) & 1u;
}

__device__ __forceinline__ int64_t gid() { return (int64_t)blockIdx.x * blockDim.x + threadIdx.x; }

// Squared distance from c to the box [lb, ub] (0 inside).
__device__ __forceinline__ float box_dist2(const float (&lb)[3], const float (&ub)[3], V3<float> c) {
  const float dx = fmaxf(fmaxf(lb[0] - c.x, c.x - ub[0]), 0.f);
  const float dy = fmaxf(fmaxf(lb[1] - c.y, c.y - ub[1]), 0.f);
  const float dz = fmaxf(fmaxf(lb[2] - c.z, c.z - ub[2]), 0.f);
  return dx * dx + dy * dy + dz * dz;
}

// Squared distance between the boxes [lb, ub] and [l, u] (0 when they meet).
__device__ __forceinline__ float box_box_dist2(const float (&lb)[3], const float (&ub)[3], V3<float> l, V3<float> u) {
  const float dx = fmaxf(fmaxf(lb[0] - u.x, l.x - ub[0]), 0.f);
  const float dy = fmaxf(fmaxf(lb[1] - u.y, l.y - ub[1]), 0.f);
  const float dz = fmaxf(fmaxf(lb[2] - u.z, l.z - ub[2]), 0.f);
  return dx * dx + dy * dy + dz * dz;
}

// Minimum / maximum of v over the wave (every lane active; wave-uniform).
__device__ __forceinline__ float wave_minf(float v) {
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) v = fminf(v, __shfl_xor(v, s, 64));
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ float wave_maxf(float v) {
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) v = fmaxf(v, __shfl_xor(v, s, 64));
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// Minimum of v over the wave (every lane active; wave-uniform result).
__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) v = min(v, __shfl_xor(v, s, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

// Maximum of v over the wave's active lanes (wave-uniform result).
__device__ __forceinline__ int wave_max_i(int v) {
  for (int m = 32; m > 0; m >>= 1) v = max(v, __shfl_xor(v, m, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

// The FP32 walk's band covers its rounding for joint values within these
// ranges (an angle's FP32 rounding is |q| 2^-24, so within 4 pi it stays
// below 1e-6 rad; a translation within 16 m, below 1e-6 m).  A state with
// a value outside them is decided by the FP64 walk.
constexpr double kFp32AngleRange = 4.0 * M_PI;
constexpr double kFp32LinearRange = 16.0;
__device__ __forceinline__ bool fp32_range_col(uint64_t rev_mask, int col, double v) {
  return fabs(v) <= (((rev_mask >> col) & 1ull) ? kFp32AngleRange : kFp32LinearRange);
}

// The kernel's one argument struct, read again from memory: a phase that takes
// its arguments through this leaves no scalar registers held (or spilled) for
// them in the phases around it.
template <class A>
__device__ __forceinline__ const A& args_again() {
#if defined(__HIP_DEVICE_COMPILE__)
  auto p = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const A*)p;
#else
  return *(const A*)nullptr;  // host pass: never executed, only type-checked
#endif
}

// The edge kernels' running time, from the device's constant-rate clock: the
// first workgroups' starts and, in as many words, the latest ends; the host
// takes the span when it is asked.  (Events around the kernel cost 7 us a call,
// 12 more where the call is then waited for.)  Also clears what the next
// launch adds to and the counts of earlier ones.  kStaged: the launch counts
// in its slot's word, otherwise in the recheck count.
template <bool kStaged>
__device__ __forceinline__ void edge_begin(const EdgeArgs& ea) {
  if (ea.clock) {
    uint64_t* mine = ea.clock + ea.slot * 2 * kEdgeClocks;
    uint64_t* next = ea.clock + (1 - ea.slot) * 2 * kEdgeClocks;
    if (blockIdx.x < kEdgeClocks && threadIdx.x == 0) mine[blockIdx.x] = (uint64_t)wall_clock64();
    if (blockIdx.x == 0)
      for (int i = threadIdx.x; i < 2 * kEdgeClocks; i += blockDim.x) next[i] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int i = 0; i < kEdgeSlots; ++i)
      if (!kStaged || i != ea.slot) ea.counter[kCntStaged + i] = 0;
    if (kStaged) ea.counter[kCntRecheck] = 0;
  }
}
// By one lane of a wave, after its last edge.
__device__ __forceinline__ void edge_clock_end(const EdgeArgs& ea) {
  if (!ea.clock) return;
  unsigned long long* end = reinterpret_cast<unsigned long long*>(ea.clock) + (ea.slot * 2 + 1) * kEdgeClocks;
  atomicMax(end + blockIdx.x % kEdgeClocks, (unsigned long long)wall_clock64());
}

// Orders a wave's own LDS accesses: what its lanes wrote before is what they
// read after.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// The lane's rank among the lanes of mask m.
__device__ __forceinline__ int lane_rank(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

// Four consecutive floats of a table read as one wave-uniform load.
struct alignas(16) Quad4 {
  float v[4];
};

// One kept tile t of cloud_block_min: the spheres' minima over its points.
template <int NK>
__device__ __forceinline__ void cloud_tile_min(const SceneArgs<float>& sc, int t, const CloudTile& T,
                                               const V3<float> (&c)[NK], int n,
                                               float (&best)[NK]) {
  V3<float> cl[NK];
  float tb[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    cl[k] = V3<float>{c[k].x - T.o[0], c[k].y - T.o[1], c[k].z - T.o[2]};
    tb[k] = FLT_MAX;
  }
  const Quad4* Bt = reinterpret_cast<const Quad4*>(sc.tileB + (int64_t)t * 4 * kCloudTile);
  for (int m = 0; m < 4; ++m) {
    for (int j4 = 0; j4 < 4; ++j4) {
      // points 16 m + 4 j4 .. + 3: components x, y, z, |p'|^2
      const Quad4 X = cload(Bt, m * 16 + 0 * 4 + j4), Y = cload(Bt, m * 16 + 1 * 4 + j4);
      const Quad4 Z = cload(Bt, m * 16 + 2 * 4 + j4), W = cload(Bt, m * 16 + 3 * 4 + j4);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
#pragma unroll
        for (int k = 0; k < NK; ++k) {
          if (k < n)
            tb[k] = fminf(tb[k], fmaf(X.v[jj], cl[k].x, fmaf(Y.v[jj], cl[k].y, fmaf(Z.v[jj], cl[k].z, W.v[jj]))));
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NK; ++k) best[k] = fminf(best[k], tb[k] + dot(cl[k], cl[k]));
}

// Per sphere k < n of a block, min |c_k - p|^2 over the points of cloud oc
// that lie in tiles within sqrt(reach2) of the block's bounding centre g
// (FLT_MAX when none).  Super-tiles, then tiles, are skipped for the whole
// wave when no `live` lane's g reaches their box: 64 of them at a time are
// first tested against the box around the live lanes' g, a box a lane, and
// the survivors of that ballot are tested lane by lane.  A kept tile's points
// are compared in tile-local coordinates, |c - p|^2 = |c'|^2 + (|p'|^2 -
// 2 c'.p'), from the matrix-core pass's operands (-2 p', |p'|^2).
template <int NK>
__device__ __forceinline__ void cloud_block_min(const SceneArgs<float>& sc, int oc, const V3<float> (&c)[NK],
                                                int n, V3<float> g, float reach2, bool live,
                                                float (&best)[NK]) {
#pragma unroll
  for (int k = 0; k < NK; ++k) best[k] = FLT_MAX;
  if (!wave_any(live)) return;
  const V3<float> gl{wave_minf(live ? g.x : FLT_MAX), wave_minf(live ? g.y : FLT_MAX), wave_minf(live ? g.z : FLT_MAX)};
  const V3<float> gu{wave_maxf(live ? g.x : -FLT_MAX), wave_maxf(live ? g.y : -FLT_MAX),
                     wave_maxf(live ? g.z : -FLT_MAX)};
  const int lane = threadIdx.x & 63;
  const int s_end = sc.super_at[oc + 1];
  for (int s0 = sc.super_at[oc]; s0 < s_end; s0 += 64) {
    bool snear = false;
    if (s0 + lane < s_end) {
      const CloudSuper Sv = sc.supers[s0 + lane];  // a super-tile a lane: vector loads
      snear = box_box_dist2(Sv.lb, Sv.ub, gl, gu) <= reach2;
    }
    for (uint64_t smask = __ballot(snear); smask; smask &= smask - 1) {
      const CloudSuper S = cload(sc.supers, s0 + __builtin_ctzll(smask));
      if (!wave_any(live && box_dist2(S.lb, S.ub, g) <= reach2)) continue;
      const int t_end = S.first + S.count;
      for (int t0 = S.first; t0 < t_end; t0 += 64) {
        bool tnear = false;
        if (t0 + lane < t_end) {
          const CloudTile Tv = sc.tiles[t0 + lane];
          tnear = box_box_dist2(Tv.lb, Tv.ub, gl, gu) <= reach2;
        }
        for (uint64_t tmask = __ballot(tnear); tmask; tmask &= tmask - 1) {
          const int t = t0 + __builtin_ctzll(tmask);
          const CloudTile T = cload(sc.tiles, t);
          if (!wave_any(live && box_dist2(T.lb, T.ub, g) <= reach2)) continue;
          cloud_tile_min<NK>(sc, t, T, c, n, best);
        }
      }
    }
  }
}

// The nearest point of cloud oc to c, per lane (an exhaustive search over
// the tiles, skipping those whose box is farther than the best so far), and
// its squared distance in best.  kNamed: with named roundings.
template <bool kNamed = false>
__device__ __forceinline__ V3<float> cloud_nearest(const SceneArgs<float>& sc, int oc, V3<float> c, float& best) {
  best = FLT_MAX;
  V3<float> bp = c;
  for (int si = sc.super_at[oc]; si < sc.super_at[oc + 1]; ++si) {
    const CloudSuper S = sc.supers[si];
    if (box_dist2(S.lb, S.ub, c) > best) continue;
    for (int t = S.first; t < S.first + S.count; ++t) {
      const CloudTile T = sc.tiles[t];
      if (box_dist2(T.lb, T.ub, c) > best) continue;
      const V3<float> cl{c.x - T.o[0], c.y - T.o[1], c.z - T.o[2]};
      const float off = kNamed ? dot3(cl, cl) : dot(cl, cl);
      const float* Bt = sc.tileB + (int64_t)t * 4 * kCloudTile;
      for (int j = 0; j < kCloudTile; ++j) {
        const float* col = Bt + (j / 16) * 64 + (j % 16);
        const float bx = col[0], by = col[16], bz = col[32], bw = col[48];
        const float d2 = fmaf(bx, cl.x, fmaf(by, cl.y, fmaf(bz, cl.z, bw))) + off;
        if (d2 < best) {
          best = d2;
          bp = V3<float>{T.o[0] - 0.5f * bx, T.o[1] - 0.5f * by, T.o[2] - 0.5f * bz};
        }
      }
    }
  }
  return bp;
}

// The base's own q columns (a planar or floating base), as (column, axis,
// origin) frames: translations along x, y, z, then the roll / pitch / yaw
// axes of the base's Rz(yaw) Ry(pitch) Rx(roll) rotation.
template <class QS, class F>
__device__ __forceinline__ void base_columns(const KinArgs<float>& ka, const Pose<float>& base, const QS& qs, F&& f) {
  const int n = ka.n_q_cols;
  if (ka.base_type == PMP_BASE_PLANAR) {
    f(n, V3<float>{1.f, 0.f, 0.f}, base.t);
    f(n + 1, V3<float>{0.f, 1.f, 0.f}, base.t);
    f(n + 2, V3<float>{0.f, 0.f, 1.f}, base.t);
  } else if (ka.base_type == PMP_BASE_FLOATING) {
    const float pitch = (float)qs.get(n + 4), yaw = (float)qs.get(n + 5);
    float sp, cp, sy, cy;
    sincosf(pitch, &sp, &cp);
    sincosf(yaw, &sy, &cy);
    f(n, V3<float>{1.f, 0.f, 0.f}, base.t);
    f(n + 1, V3<float>{0.f, 1.f, 0.f}, base.t);
    f(n + 2, V3<float>{0.f, 0.f, 1.f}, base.t);
    f(n + 3, V3<float>{cy * cp, sy * cp, -sp}, base.t);  // Rz(yaw) Ry(pitch) x
    f(n + 4, V3<float>{-sy, cy, 0.f}, base.t);           // Rz(yaw) y
    f(n + 5, V3<float>{0.f, 0.f, 1.f}, base.t);
  }
}

}  // namespace pmp
