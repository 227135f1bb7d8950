// Validity tests of staged workgroups (stage.hpp), shared by the batch of
// configurations and the motion check: what the waves of a workgroup do with
// the staged poses.
//
// The waves take slices (a run of one sphere block's candidate primitives),
// self pairs and, with clouds, a few spheres of a block from a queue and test
// them in FP32.  A test decided outside the band marks the configuration
// as colliding, and later items skip it; a test inside the band is put on the
// workgroup's pending list as the one (sphere, primitive), (sphere, cloud) or
// (sphere, sphere) pair it concerns.  At the end the first wave re-decides the
// pending pairs of configurations not yet colliding in FP64, a lane per pair:
// every other pair was decided outside the band, so the pairs decide the
// configuration.  A configuration the FP32 walk cannot decide at all (joint
// values outside its ranges, a rotation outside the cull table's bounds, NaN
// centres, a full pending list) is walked in FP64 whole.
//
// Sphere-vs-cloud queries (spheres inside the cloud's AABB pre-test) are
// answered one at a time by all lanes of a wave: 64
// super-tiles, then the tiles of four surviving super-tiles, then 64 points a
// step, stopping at the first point certainly inside.
#pragma once

#include <float.h>

#include <type_traits>

#include "stage.hpp"

namespace pmp {

// Per configuration: a certain collision; FP64 decides all of it; FP64 decided
// it or a pending pair of it.
enum ValidFlag { kHit = 1, kWhole = 2, kPended = 4 };
constexpr int kPendMax = 64;     // pending pairs a workgroup keeps

// The workgroup's results under way, in LDS.  kFirst: its configurations are
// the states of one motion in visiting order and only the first colliding one
// matters, so those past the first certain collision count as decided.
template <bool kFirst>
struct ValidLds {
  int* flags;  // [C]
  int* first;  // kFirst: the first certain collision
  int* pend;   // [3][kPendMax]: configuration, sphere, primitive (>= 0, kind-sorted) or -1 - second sphere
  int* count;  // pending pairs
  __device__ __forceinline__ void mark(int cfg, int f) const {
    atomicOr(flags + cfg, f);
    if (kFirst && (f & kHit)) atomicMin(first, cfg);
  }
  __device__ __forceinline__ int state(int cfg) const {
    int f = *reinterpret_cast<volatile int*>(flags + cfg);
    if (kFirst && cfg > *reinterpret_cast<volatile int*>(first)) f |= kHit;
    return f;
  }
  __device__ __forceinline__ void defer(int cfg, int sphere, int other) const {
    const int i = atomicAdd(count, 1);
    if (i < kPendMax) {
      pend[i] = cfg;
      pend[kPendMax + i] = sphere;
      pend[2 * kPendMax + i] = other;
    } else {
      mark(cfg, kWhole);
    }
  }
};

// One sphere against a cloud, by the whole wave: 1 when some point is
// certainly inside R = r + rc, 2 when one may be (within the band, widened by
// the tile-local form's error), else 0 (CloudSDF::is_outside,
// primitive_sdf.hpp:597-603: collide iff min |c - p|^2 <= R^2).
__device__ __forceinline__ int cloud_query(const SceneArgs<float>& sc, int oc, V3<float> c, float R, float band,
                                           int lane) {
  const float R2 = R * R, w = band * (2.0f * R + band), cap = (R + band) * (R + band);
  int res = 0;
  const int s_end = sc.super_at[oc + 1];
  for (int s0 = sc.super_at[oc]; s0 < s_end; s0 += 64) {
    bool near = false;
    int first = 0, count = 0;
    if (s0 + lane < s_end) {
      const CloudSuper S = sc.supers[s0 + lane];
      near = box_dist2(S.lb, S.ub, c) <= cap;
      first = S.first;
      count = S.count;
    }
    uint64_t smask = __ballot(near);
    while (smask) {
      // the tiles of up to four super-tiles, sixteen lanes each
      int tile = -1;
#pragma unroll
      for (int u = 0; u < 64 / kCloudSuper; ++u) {
        const int j = smask ? __builtin_ctzll(smask) : 0;
        const int f = __builtin_amdgcn_readlane(first, j), n = smask ? __builtin_amdgcn_readlane(count, j) : 0;
        smask &= smask - 1;
        if (lane / kCloudSuper == u && lane % kCloudSuper < n) tile = f + lane % kCloudSuper;
      }
      bool tnear = false;
      if (tile >= 0) {
        const CloudTile T = sc.tiles[tile];
        tnear = box_dist2(T.lb, T.ub, c) <= cap;
      }
      for (uint64_t tmask = __ballot(tnear); tmask; tmask &= tmask - 1) {
        const int t = __builtin_amdgcn_readlane(tile, __builtin_ctzll(tmask));
        const CloudTile T = cload(sc.tiles, t);
        const float* col = sc.tileB + (int64_t)t * 4 * kCloudTile + (lane >> 4) * 64 + (lane & 15);
        const V3<float> cl{c.x - T.o[0], c.y - T.o[1], c.z - T.o[2]};
        const float off = dot(cl, cl);
        const float d2 = fmaf(col[0], cl.x, fmaf(col[16], cl.y, fmaf(col[32], cl.z, col[48]))) + off;
        const float err = kCloudGemmErr * (off + tile_rho2(T));
        if (__any(d2 + err - R2 < -w)) return 1;
        if (__any(!(d2 - err - R2 > w))) res = 2;
      }
    }
  }
  return res;
}

// The cull table assumes |q|^2 of a rotation within [n2_lo, n2_hi] (so that
// |R v| <= grow |v|), and with a finite translation no centre of such a rotation
// is NaN; any other configuration is left to the FP64 walk.
__device__ __forceinline__ bool sound_pose(const Pose<float>& P, float n2_lo, float n2_hi) {
  const float n2 = P.q.x * P.q.x + P.q.y * P.q.y + P.q.z * P.q.z + P.q.w * P.q.w;
  return n2 >= n2_lo && n2 <= n2_hi && fabsf(P.t.x) <= FLT_MAX && fabsf(P.t.y) <= FLT_MAX && fabsf(P.t.z) <= FLT_MAX;
}

// One slice of block candidates for the configurations still `live`.
template <int H, bool kFirst>
__device__ __forceinline__ void valid_slice(const Stage<H>& S, const KinArgs<float>& ka, const SceneArgs<float>& sc,
                                            const DevCullSlice& it, float band, const ValidLds<kFirst>& out) {
  constexpr int NK = Stage<H>::NK;
  bool live = (out.state(S.cfg) & (kHit | kWhole)) == 0;
  if (!wave_any(live)) return;
  const DevSphereBlock bk = cload(ka.blocks, it.block);
  const Pose<float> P = S.pose(bk.pose);
  const M3<float> R = qmat(P.q);
  if (live && !sound_pose(P, bk.n2_lo, bk.n2_hi)) {
    out.mark(S.cfg, kWhole);
    live = false;
  }
  const float growf = 1.0f + 2.0f * fmaxf(0.0f, fmaxf(bk.n2_hi - 1.0f, 1.0f - bk.n2_lo)) + 1e-6f;
  const float reach = bk.G * growf + band + 1e-4f;
  V3<float> c[NK];
  float r[NK];
  int n;
  S.spheres(ka, it.block, bk, P, R, c, r, n);
  auto sphere_of = [&](int k) {
    return H == 1 ? cload(ka.blocks[it.block].sph, k) : ka.blocks[it.block].sph[S.sub * NK + k];
  };
  const V3<float> g = add(mv(R, V3<float>{bk.g[0], bk.g[1], bk.g[2]}), P.t);
  const CullRange cr = cload(sc.cull_range, it.block);
  const DevPrim<float>* vp = reinterpret_cast<const DevPrim<float>*>(sc.vprims);
  auto kind = [&](auto kc) {
    constexpr int K = decltype(kc)::value;
    const int hi = min(it.hi, cr.at[K + 1]);
    for (int i = max(it.lo, cr.at[K]); i < hi; ++i) {
      const CullEntry ce = cload(sc.cull, i);
      // every member sphere is outside the primitive's AABB inflated by its
      // radius plus the band when the bounding centre is outside the grown box
      const bool near = live && !(g.x < ce.lb[0] || g.x > ce.ub[0] || g.y < ce.lb[1] || g.y > ce.ub[1] ||
                                  g.z < ce.lb[2] || g.z > ce.ub[2]);
      if (!wave_any(near)) continue;
      const DevPrim<float> Q = cload(vp, ce.prim);
      if constexpr (K != kKindGround) {  // the ground's test is not a pure distance
        bool nb = false;
        if (!wave_any(near && collide_kind<K>(Q, g, reach, 0.0f, nb))) continue;
      }
      bool hit = false;
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        if (k < n) {
          bool inb = false;
          const bool col = collide_kind<K>(Q, c[k], r[k], band, inb);
          hit |= live && col && !inb;
          if (live && inb) out.defer(S.cfg, sphere_of(k), ce.prim);
        }
      }
      if (hit) {
        out.mark(S.cfg, kHit);
        live = false;
      }
      if (kFirst && wave_any(hit)) live = live && (out.state(S.cfg) & kHit) == 0;
      if (!wave_any(live)) return;
    }
  };
  kind(std::integral_constant<int, kKindBoxAA>{});
  kind(std::integral_constant<int, kKindBoxRot>{});
  kind(std::integral_constant<int, kKindCylZ>{});
  kind(std::integral_constant<int, kKindCylRot>{});
  kind(std::integral_constant<int, kKindSphere>{});
  kind(std::integral_constant<int, kKindGround>{});
}

// Spheres [k0, k0 + kCloudSpheres) of each lane's share of a block against the
// clouds: the lanes whose sphere is inside a cloud's AABB pre-test are answered
// one at a time by all of them.
// (4,096 motions 585 us with two spheres an item, 597 with four, 654 with eight
// and 637 with one; 512 of the Fetch-like robot 117, 133, 133 and 104.)
constexpr int kCloudSpheres = 2;
template <int H, bool kFirst>
__device__ __forceinline__ void valid_cloud(const Stage<H>& S, const KinArgs<float>& ka, const SceneArgs<float>& sc,
                                            int block, int k0, float band, const ValidLds<kFirst>& out) {
  constexpr int NK = Stage<H>::NK, G = NK < kCloudSpheres ? NK : kCloudSpheres;
  bool live = (out.state(S.cfg) & (kHit | kWhole)) == 0;
  if (!wave_any(live)) return;
  const DevSphereBlock bk = cload(ka.blocks, block);
  const Pose<float> P = S.pose(bk.pose);
  if (live && !sound_pose(P, bk.n2_lo, bk.n2_hi)) {
    out.mark(S.cfg, kWhole);
    live = false;
  }
  const M3<float> R = qmat(P.q);
  const int at = S.sub * NK + k0;
  V3<float> c[G];
  float r[G];
#pragma unroll
  for (int k = 0; k < G; ++k) {
    const Quad4 s = reinterpret_cast<const Quad4*>(ka.blocks[block].s)[at + k];
    c[k] = add(mv3(R, V3<float>{s.v[0], s.v[1], s.v[2]}), P.t);
    r[k] = s.v[3];
  }
  for (int p = sc.vrange[kKindCloud]; p < sc.vrange[kKindCloud + 1]; ++p) {
    const DevPrim<float> Pc = cload(reinterpret_cast<const DevPrim<float>*>(sc.vprims), p);
#pragma unroll
    for (int k = 0; k < G; ++k) {
      const bool ask = live && at + k < bk.n && !outside_aabb(Pc, c[k], r[k]);
      for (uint64_t m = __ballot(ask); m; m &= m - 1) {
        const int i = __builtin_ctzll(m), cfg = i & (Stage<H>::C - 1);
        if (__builtin_amdgcn_readfirstlane(out.state(cfg)) & kHit) continue;
        auto rd = [&](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i)); };
        const int res = cloud_query(sc, (Pc.flags >> 4) & 15, V3<float>{rd(c[k].x), rd(c[k].y), rd(c[k].z)},
                                    rd(r[k]) + Pc.p0, band, S.lane);
        if (S.lane == i) {
          if (res == 1) out.mark(cfg, kHit);
          if (res == 2) out.defer(cfg, ka.blocks[block].sph[at + k], p);
        }
      }
    }
  }
}

// One self pair (check_self_collision, primitive_sphere_collision.cpp:222-254).
template <int H, bool kFirst>
__device__ __forceinline__ void valid_pair(const Stage<H>& S, const KinArgs<float>& ka, int k, float band,
                                           const ValidLds<kFirst>& out) {
  bool live = (out.state(S.cfg) & (kHit | kWhole)) == 0;
  if (!wave_any(live)) return;
  const DevSelfPair pr = cload(ka.pairs, k);
  const Pose<float> P1 = S.pose(pr.pose1), P2 = S.pose(pr.pose2);
  const M3<float> R1 = qmat(P1.q), R2 = qmat(P2.q);
  const V3<float> g1 = add(mv(R1, V3<float>{pr.bound1[0], pr.bound1[1], pr.bound1[2]}), P1.t);
  const V3<float> g2 = add(mv(R2, V3<float>{pr.bound2[0], pr.bound2[1], pr.bound2[2]}), P2.t);
  const float n1 = P1.q.x * P1.q.x + P1.q.y * P1.q.y + P1.q.z * P1.q.z + P1.q.w * P1.q.w;
  const float n2 = P2.q.x * P2.q.x + P2.q.y * P2.q.y + P2.q.z * P2.q.z + P2.q.w * P2.q.w;
  const float grow = 1.0f + 2.0f * fmaxf(fabsf(n1 - 1.0f), fabsf(n2 - 1.0f));
  const V3<float> dg = sub(g1, g2);
  const float far = (pr.bound1[3] + pr.bound2[3]) * grow + band + 1e-4f;
  if (!wave_any(live && !(dot(dg, dg) > far * far * 1.0001f))) return;
  bool hit = false;
  for (int i0 = pr.begin1; i0 < pr.end1; i0 += H) {
    const int i = H == 1 ? i0 : i0 + S.sub;
    DevSphere<float> a{};
    if constexpr (H == 1)
      a = cload(ka.spheres, i);
    else if (i < pr.end1)
      a = ka.spheres[i];
    const V3<float> ci = add(mv(R1, V3<float>{a.x, a.y, a.z}), P1.t);
    for (int j = pr.begin2; j < pr.end2; ++j) {
      const DevSphere<float> bb = cload(ka.spheres, j);
      const V3<float> d = sub(ci, add(mv(R2, V3<float>{bb.x, bb.y, bb.z}), P2.t));
      const float rs = a.r + bb.r, m = dot(d, d) - rs * rs;
      const bool inb = !(fabsf(m) > band * (2.0f * rs + band));  // NaN too
      if (i < pr.end1 && live) {
        if (inb) out.defer(S.cfg, i, -1 - j);
        hit |= !inb && m < 0.0f;
      }
    }
  }
  if (hit) out.mark(S.cfg, kHit);
}

// Whether a workgroup of W waves takes slices of the blocks' candidates or,
// sparing the repeated set-up, whole blocks: slices while there are too few
// blocks and self pairs to balance it.  (48 primitives: 7R arm, 8 blocks, 16,384
// configurations with 16 waves 17.7 us by slices, 22.5 by blocks; 131,072 with 4
// waves 60 and 57; 14 joints and self pairs, 16,384 42 and 38; Fetch-like, 16
// primitives, 100,003 94 and 90; 1,024 motions of the 14-joint robot 96 and 90.)
inline bool slice_blocks(const KinArgs<float>& ka, int W) { return ka.n_units < 2 * W; }

// The items of a workgroup: slices, self pairs, then some spheres of a block
// against the clouds, whose configurations the cheaper tests may have decided.
template <bool kCloud, int H, bool kFirst>
__device__ __forceinline__ void valid_items(const Stage<H>& S, const KinArgs<float>& ka, const SceneArgs<float>& sc,
                                            float band, const ValidLds<kFirst>& out, int* queue, bool sliced) {
  constexpr int G = Stage<H>::NK < kCloudSpheres ? 1 : Stage<H>::NK / kCloudSpheres;  // cloud items of a block
  const int n_blocks = ka.n_units - ka.n_pairs, n_ext = sc.n_prims == 0 ? 0 : (sliced ? sc.n_slices : n_blocks);
  const int n_solid = n_ext + ka.n_pairs, n_items = n_solid + (kCloud ? n_blocks * G : 0);
  for (;;) {
    int it = 0;
    if (S.lane == 0) it = atomicAdd(queue, 1);
    it = __builtin_amdgcn_readfirstlane(it);
    if (it >= n_items) break;
    if (it < n_ext)
      valid_slice(S, ka, sc, sliced ? cload(sc.slices, it) : DevCullSlice{n_blocks - 1 - it, 0, INT_MAX, 0}, band, out);
    else if (!kCloud || it < n_solid)
      valid_pair(S, ka, it - n_ext, band, out);
    else if constexpr (kCloud)
      valid_cloud(S, ka, sc, (it - n_solid) / G, (it - n_solid) % G * kCloudSpheres, band, out);
  }
}

// A point cloud against one sphere in FP64, by the whole wave (uniform
// arguments): CloudSDF::is_outside after the AABB pre-test, the minimum taken
// over the tiles that can reach within r + rc.
__device__ __forceinline__ bool cloud_hit64(const SceneArgs<double>& sc, const DevPrim<double>& P, V3<double> c, double r,
                                            int lane) {
  const double R = r + P.p0, lim = R * R * (1.0 + 1e-12) + 1e-300;
  auto far = [&](auto& lb, auto& ub) {
    const double dx = fmax(fmax((double)lb[0] - c.x, c.x - (double)ub[0]), 0.0);
    const double dy = fmax(fmax((double)lb[1] - c.y, c.y - (double)ub[1]), 0.0);
    const double dz = fmax(fmax((double)lb[2] - c.z, c.z - (double)ub[2]), 0.0);
    return dx * dx + dy * dy + dz * dz > lim;
  };
  double best = DBL_MAX;
  const int oc = (P.flags >> 4) & 15;
  for (int s0 = sc.super_at[oc]; s0 < sc.super_at[oc + 1]; s0 += 64) {
    bool near = false;
    if (s0 + lane < sc.super_at[oc + 1]) {
      const CloudSuper S = sc.supers[s0 + lane];
      near = !far(S.lb, S.ub);
    }
    for (uint64_t smask = __ballot(near); smask; smask &= smask - 1) {
      const CloudSuper S = cload(sc.supers, s0 + __builtin_ctzll(smask));
      bool tnear = false;
      if (lane < S.count) {
        const CloudTile64 T = sc.tiles64[S.first + lane];
        tnear = !far(T.lb, T.ub);
      }
      for (uint64_t tmask = __ballot(tnear); tmask; tmask &= tmask - 1) {
        const double* pt = sc.pts64 + ((int64_t)(S.first + __builtin_ctzll(tmask)) * kCloudTile + lane) * 4;
        const double ex = pt[0] - c.x, ey = pt[1] - c.y, ez = pt[2] - c.z;
        best = fmin(best, ex * ex + ey * ey + ez * ez);
      }
    }
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) best = fmin(best, __shfl_xor(best, s, 64));
  return !(sqrt(best) - P.p0 > r);
}

__device__ __forceinline__ double readlane64(double v, int i) {
  const long long u = __builtin_bit_cast(long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, i);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), i);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Cloud `P` (wave-uniform) against the spheres of the lanes that `ask`, one
// lane at a time; whether this lane's collides.
__device__ __forceinline__ bool cloud_hits64(const SceneArgs<double>& sc, const DevPrim<double>& P, V3<double> c, double r,
                                             bool ask, int lane) {
  bool hit = false;
  for (uint64_t m = __ballot(ask && !outside_aabb(P, c, r)); m; m &= m - 1) {
    const int i = __builtin_ctzll(m);
    const bool h = cloud_hit64(sc, P, V3<double>{readlane64(c.x, i), readlane64(c.y, i), readlane64(c.z, i)},
                               readlane64(r, i), lane);
    if (lane == i) hit = h;
  }
  return hit;
}

// FP64 walk that keeps the poses of two nodes per lane.
struct TwoPoses64 {
  static constexpr bool kSelf = false;
  static constexpr bool kBlocks = true;
  int node1, node2;
  bool idle;
  Pose<double> P1{}, P2{};
  int last = -1;
  __device__ bool alive() const { return !idle && last < max(node1, node2); }
  template <class QS>
  __device__ void begin(const Pose<double>&, const QS&) {}
  __device__ void node(int n, const DevNode<double>&, const Pose<double>& P) {
    if (n == node1) P1 = P;
    if (n == node2) P2 = P;
    last = n;
  }
  __device__ void sphere(int, V3<double>, double) {}
  __device__ void blocks(const DevNode<double>&, const Pose<double>&) {}
  __device__ void self(const DevSelfPair&, int, int, V3<double>, V3<double>, double) {}
};

// FP64 walk of whole configurations with the reference's own tests: per
// primitive-checked sphere the AABB pre-test and is_outside, per self pair
// the strict squared-distance test.  The group-sphere broad phase of the
// reference only culls, so it is not needed for the result.  The waves share
// the sphere blocks and self pairs and the lanes of a configuration a block's
// spheres (lane `part` takes nk of them).  A block's candidates are those of
// the FP32 pass: its grown boxes carry a 1e-4 m slack, far above the FP32/FP64
// centre difference, so a candidate they drop is outside the AABB pre-test in
// FP64 too.
template <bool kFirst>
struct WholeVis64 {
  static constexpr bool kSelf = true;
  static constexpr bool kRanged = true;
  static constexpr bool kBlocks = true;
  const KinArgs<double>& ka;
  const SceneArgs<double>& sc;
  const ValidLds<kFirst>& out;
  int lane, cfg, part, nk, wave, n_waves;
  bool collided;  // or decided by another wave, or nothing to do
  __device__ bool alive() const { return !collided; }
  __device__ int last_node() const { return ka.n_nodes - 1; }
  __device__ int pair_lo() const { return ka.n_pairs * wave / n_waves; }
  __device__ int pair_hi() const { return ka.n_pairs * (wave + 1) / n_waves; }
  template <class QS>
  __device__ void begin(const Pose<double>&, const QS&) {}
  __device__ void node(int, const DevNode<double>&, const Pose<double>&) {}
  __device__ void sphere(int, V3<double>, double) {}
  // Candidates i0 + (bits of mask) of kind K.
  template <int K>
  __device__ __forceinline__ void kind(V3<double> c, double r, bool has, int i0, uint64_t mask, int lo, int hi,
                                       bool nocull) {
    lo = max(lo - i0, 0);
    hi = min(hi - i0, 64);
    if (lo >= hi) return;
    mask &= (~0ull << lo) & (~0ull >> (64 - hi));
    for (; mask; mask &= mask - 1) {
      if (!wave_any(has && !collided)) return;
      const int i = i0 + __builtin_ctzll(mask);
      const DevPrim<double> P =
          cload(reinterpret_cast<const DevPrim<double>*>(sc.vprims), nocull ? i : cload(sc.cull, i).prim);
      if (has && !collided && !outside_aabb(P, c, r) && !is_outside_ref<double, K>(P, c, r)) collided = true;
    }
  }
  __device__ __forceinline__ void block(int bi, const Pose<double>& P, const M3<double>& R, bool nocull) {
    const DevSphereBlock bk = cload(ka.blocks, bi);
    auto centre = [&](int k, bool& has, double& r) {
      const int at = part * nk + k;
      has = at < bk.n;
      const DevSphere<double> sp = ka.spheres[ka.blocks[bi].sph[has ? at : 0]];
      r = sp.r;
      return add(mv(R, V3<double>{sp.x, sp.y, sp.z}), P.t);
    };
    bool has;
    double r;
    for (int k = 0; k < nk; ++k) {
      const V3<double> c = centre(k, has, r);
      // a NaN centre collides with every primitive but a cloud, whose nearest
      // point then decides (nothing is nearer than infinity: it does not)
      if (has && sc.vrange[kKindCloud] > 0 && is_nan3(c)) collided = true;
      for (int p = sc.vrange[kKindCloud]; p < sc.vrange[kKindCloud + 1]; ++p)
        if (cloud_hits64(sc, cload(reinterpret_cast<const DevPrim<double>*>(sc.vprims), p), c, r, has && !collided,
                         lane))
          collided = true;
    }
    const V3<double> g = add(mv(R, V3<double>{bk.g[0], bk.g[1], bk.g[2]}), P.t);
    const CullRange cr = cload(sc.cull_range, bi);
    auto at = [&](int k) { return nocull ? sc.vrange[k] : cr.at[k]; };
    for (int i0 = at(0); i0 < at(kKindCloud); i0 += 64) {
      uint64_t mask = 0;
      for (int i = i0; i < min(i0 + 64, at(kKindCloud)); ++i) {
        bool near = !collided;
        if (!nocull) {
          const CullEntry ce = cload(sc.cull, i);
          near = near && !(g.x < ce.lb[0] || g.x > ce.ub[0] || g.y < ce.lb[1] || g.y > ce.ub[1] || g.z < ce.lb[2] ||
                           g.z > ce.ub[2]);
        }
        if (wave_any(near)) mask |= 1ull << (i - i0);
      }
      if (mask == 0) continue;
      for (int k = 0; k < nk; ++k) {
        const V3<double> c = centre(k, has, r);
        kind<kKindBoxAA>(c, r, has, i0, mask, at(kKindBoxAA), at(kKindBoxAA + 1), nocull);
        kind<kKindBoxRot>(c, r, has, i0, mask, at(kKindBoxRot), at(kKindBoxRot + 1), nocull);
        kind<kKindCylZ>(c, r, has, i0, mask, at(kKindCylZ), at(kKindCylZ + 1), nocull);
        kind<kKindCylRot>(c, r, has, i0, mask, at(kKindCylRot), at(kKindCylRot + 1), nocull);
        kind<kKindSphere>(c, r, has, i0, mask, at(kKindSphere), at(kKindSphere + 1), nocull);
        kind<kKindGround>(c, r, has, i0, mask, at(kKindGround), at(kKindGround + 1), nocull);
      }
    }
  }
  __device__ __forceinline__ void blocks(const DevNode<double>& nd, const Pose<double>& P) {
    if (nd.block_begin >= nd.block_end) return;
    if (out.state(cfg) & kHit) collided = true;
    const M3<double> R = qmat(P.q);
    // outside the norm bounds the cull table assumed: test every primitive
    const double n2 = P.q.x * P.q.x + P.q.y * P.q.y + P.q.z * P.q.z + P.q.w * P.q.w;
    const bool nocull = wave_any(alive() && !(n2 >= nd.n2_lo && n2 <= nd.n2_hi));
    for (int bi = nd.block_begin; bi < nd.block_end; ++bi)
      if (bi % n_waves == wave && wave_any(alive())) block(bi, P, R, nocull);
  }
  __device__ void self(const DevSelfPair&, int, int, V3<double> ci, V3<double> cj, double rs) {
    const V3<double> d = sub(ci, cj);
    if (dot(d, d) < rs * rs) collided = true;
  }
};

// FP64 decision of what the FP32 items left open.  point(cfg) is the
// joint-value source of a configuration.  The kept poses of the walks take the
// workgroup's LDS from its start: the results lie past it.  Both return whether
// this lane decided anything.
//
// The pending pairs of configurations not yet colliding, by the first wave, a
// lane each.
template <bool kFirst, class F>
__device__ __forceinline__ bool decide_pending(int lane, int cfg, const KinArgs<float>& ka, const KinArgs<double>& k64,
                                               const SceneArgs<double>& s64, bool taylor, const ValidLds<kFirst>& out,
                                               F&& point) {
  const int n_pend = min(*out.count, kPendMax);
  if (n_pend == 0) return false;
  const int pc = lane < n_pend ? out.pend[lane] : 0, s1 = lane < n_pend ? out.pend[kPendMax + lane] : 0,
            other = lane < n_pend ? out.pend[2 * kPendMax + lane] : 0;
  const bool has = lane < n_pend && (out.state(pc) & (kHit | kWhole)) == 0;
  const int s2 = other < 0 ? -1 - other : s1;
  TwoPoses64 v{has ? ka.meta[s1].node : 0, has ? ka.meta[s2].node : 0, !has};
  run_fk(k64, point(has ? pc : cfg), taylor, v);
  const DevSphere<double> a = k64.spheres[s1];
  const V3<double> c1 = add(mv(qmat(v.P1.q), V3<double>{a.x, a.y, a.z}), v.P1.t);
  bool hit = false;
  bool cloud = false;
  if (has && other < 0) {
    const DevSphere<double> bb = k64.spheres[s2];
    const V3<double> d = sub(c1, add(mv(qmat(v.P2.q), V3<double>{bb.x, bb.y, bb.z}), v.P2.t));
    const double rs = a.r + bb.r;
    hit = dot(d, d) < rs * rs;
  } else if (has) {
    cloud = other >= s64.vrange[kKindCloud];
    const DevPrim<double>& P = reinterpret_cast<const DevPrim<double>*>(s64.vprims)[other];
    hit = !cloud && !outside_aabb(P, c1, a.r) && !is_outside_ref<double>(P, c1, a.r);
  }
  for (int p = s64.vrange[kKindCloud]; p < s64.vrange[kKindCloud + 1]; ++p)
    hit |= cloud_hits64(s64, cload(reinterpret_cast<const DevPrim<double>*>(s64.vprims), p), c1, a.r,
                        cloud && other == p, lane);
  if (has) out.mark(pc, kPended | (hit ? kHit : 0));
  wave_lds_order();
  return has;
}

// Whether some configuration is left to the FP64 walk whole: the same in every
// wave, also while the first one decides pending pairs.
template <bool kFirst>
__device__ __forceinline__ bool any_whole(const ValidLds<kFirst>& out, int cfg) {
  return wave_any((*reinterpret_cast<volatile int*>(out.flags + cfg) & kWhole) != 0);
}
// Whole configurations, by the first n_waves waves (whose kept poses fit the
// tables' LDS), nk = kBlockSpheres / H spheres of a block to each of a
// configuration's H lanes.  Configurations eight turns out of range: 1,000 of the
// 7R arm 25 us, 50,000 of it 75, of the 14-joint robot 327, of a floating 31-joint
// one 465.  (By one wave, a lane a configuration and every sphere against every
// primitive: 249, 273, 1,364 and 1,508; in a launch of their own with a lane a
// configuration: 102, 117, 414 and 454.)
template <bool kFirst, class F>
__device__ __forceinline__ bool decide_whole(int lane, int cfg, int part, int nk, int wave, int n_waves,
                                             const KinArgs<double>& k64, const SceneArgs<double>& s64, bool taylor,
                                             bool active, const ValidLds<kFirst>& out, F&& point) {
  const int f = out.state(cfg);
  const bool whole = active && (f & kWhole) && !(f & kHit) && wave < n_waves;
  if (wave_any(whole)) {
    WholeVis64<kFirst> v{k64, s64, out, lane, cfg, part, nk, wave, n_waves, !whole};
    run_fk(k64, point(cfg), taylor, v);
    if (whole) out.mark(cfg, kPended | (v.collided ? kHit : 0));
  }
  return whole;
}

// The waves of a workgroup of W whose FP64 kept poses fit lds bytes.
inline int whole_waves(const KinArgs<double>& k64, size_t lds, int W) {
  const int64_t fit = k64.slot_wave_bytes > 0 ? (int64_t)lds / k64.slot_wave_bytes : W;
  return fit < 1 ? 1 : (fit < W ? (int)fit : W);
}

}  // namespace pmp
