// Evaluate rows (value and Jacobian row of the external and of the self
// constraint per configuration) and trajectory smoothness, by staged
// workgroups (stage.hpp).
//
// evaluate_ext_collision / evaluate_self_collision
// (constraints/primitive_sphere_collision.cpp:256-383): the external value is
// the minimum over every (sphere, primitive) pair below the 0.1 m cutoff, ties
// to the smallest (group, primitive, sphere) key; the self value the minimum
// over the self pairs, ties to the first in visiting order.
//
// The waves of a workgroup take slices (a run of one sphere block's candidate
// primitives) and self pairs from a queue.  The best (value, tie key) of every
// configuration is one 64-bit word in LDS, lowered by atomic minimum: the
// order in which the waves finish decides only what is skipped, never the
// result.  A candidate is first tested, for the block's bounding sphere and
// then sphere by sphere, by a distance bound without correctly rounded roots;
// only the few (configuration, sphere) pairs that may improve on the best are
// compacted through LDS and evaluated, so the exact evaluation runs with full
// waves although nearby configurations rarely agree on what is close.  Then a
// wave per primitive type (and one for the self pair) forms the winners'
// centres and directions, and all waves write the rows' columns.
#include <type_traits>

#include "last_launch.hpp"
#include "stage.hpp"

namespace pmp {

constexpr int kWinWords = 21;  // c0, g0, mask 0; c1, c2, n, masks 1 and 2

struct StagedOut {
  float* vals;  // [cst_dim][B]
  float* jac;   // [cst_dim][D][B]
  // trajectories (offsets == nullptr: plain evaluate)
  const int64_t* offsets;
  int n_traj;
  const double* w2;
  float* cost;
  float* grad;
  int n_chunks;  // workgroups of configurations; those after them take trajectories' costs
  int sliced;    // candidates taken by slices (else by whole blocks)
  int scratch, best;  // LDS offsets (floats)
};

// The best of a configuration: the value as an unsigned integer of the same
// order in the high word, the tie key in the low word.
typedef unsigned long long Best;
__device__ __forceinline__ uint32_t ordered(float v) {
  const uint32_t u = (uint32_t)__float_as_int(v);
  return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ __forceinline__ float unordered(uint32_t u) {
  return __int_as_float((int)(u ^ ((u >> 31) ? 0x80000000u : 0xffffffffu)));
}
__device__ __forceinline__ Best no_winner() { return ((Best)ordered(kCutoff) << 32) | 0xffffffffu; }
__device__ __forceinline__ bool has_winner(Best b) { return b != no_winner(); }
__device__ __forceinline__ float best_value(Best b) { return unordered((uint32_t)(b >> 32)); }
// v below the cutoff (NaN never is)
__device__ __forceinline__ void offer(Best* best, float v, uint32_t key) {
  if (v < kCutoff) atomicMin(best, ((Best)ordered(v + 0.0f) << 32) | key);  // -0 and 0 tie
}
// The value reached so far, read while other waves lower it.
__device__ __forceinline__ float bound_of(const Best* best) {
  return unordered(reinterpret_cast<const volatile uint32_t*>(best)[1]);
}

// Keys: external (group * n_prims + primitive) * n_spheres + sphere (group
// order; fewer groups than spheres, so below n_spheres^2 n_prims); self: pair,
// then the spheres' positions in their groups.
constexpr int kSelfPosBits = 11;

// Entries a wave collects before it evaluates them: the sphere's centre and
// radius, its key and its configuration.
constexpr int kEntryWords = 6;

// Lanes a configuration has at least in scenes with clouds.
constexpr int kCloudLanes = 4;

// One slice of block candidates.
// kBoxes: candidates are first tested against their grown box (coherent
// batches, where it drops most of them before their primitive is read).
template <int H, bool kBoxes>
__device__ __forceinline__ void ext_slice(const Stage<H>& S, const KinArgs<float>& ka, const SceneArgs<float>& sc,
                                          const DevCullSlice& it, Best* best, float* entries) {
  constexpr int NK = Stage<H>::NK;
  const DevSphereBlock bk = cload(ka.blocks, it.block);
  const Pose<float> P = S.pose(bk.pose);
  const M3<float> R = qmat(P.q);
  // outside the norm bounds the cull table assumed: every primitive is a
  // candidate, and the block's first slice takes them all
  const float n2 = P.q.x * P.q.x + P.q.y * P.q.y + P.q.z * P.q.z + P.q.w * P.q.w;
  const bool all = wave_any(!(n2 >= bk.n2_lo && n2 <= bk.n2_hi));
  if (all && !it.first) return;
  const float growf = 1.0f + 2.0f * fmaxf(0.0f, fmaxf(bk.n2_hi - 1.0f, 1.0f - bk.n2_lo)) + 1e-6f;
  const float ereach = bk.G * growf + 1e-4f;
  V3<float> c[NK];
  float r[NK];
  uint32_t skey[NK];
  int n;
  S.spheres(ka, it.block, bk, P, R, c, r, n);
  // a sphere's part of the key: kept per lane with H > 1, else read when
  // wanted (eight more scalar registers would be spilled)
  auto sphere_key = [&](int group, int out) {
    return (uint32_t)group * (uint32_t)sc.n_prims * (uint32_t)ka.n_spheres + (uint32_t)out;
  };
  if constexpr (H > 1) {
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const DevSphereBlock& pb = ka.blocks[it.block];
      skey[k] = sphere_key(pb.group[S.sub * NK + k], pb.out[S.sub * NK + k]);
    }
  }
  auto key_of = [&](int k) {
    if constexpr (H > 1) return skey[k];
    const DevSphereBlock* pb = ka.blocks + it.block;
    return sphere_key(cload(pb->group, k), cload(pb->out, k));
  };
  const V3<float> g = add(mv(R, V3<float>{bk.g[0], bk.g[1], bk.g[2]}), P.t);
  const CullRange cr = cload(sc.ecull_range, it.block);
  const DevPrim<float>* vp = reinterpret_cast<const DevPrim<float>*>(sc.vprims);
  auto kind = [&](auto kc) {
    constexpr int K = decltype(kc)::value;
    const int lo = all ? sc.vrange[K] : max(it.lo, cr.at[K]), hi = all ? sc.vrange[K + 1] : min(it.hi, cr.at[K + 1]);
    for (int i = lo; i < hi; ++i) {
      int p, orig;
      if (all) {
        p = i;
        orig = cload(sc.vorig, i);
      } else {
        const CullEntry ce = cload(sc.ecull, i);
        if constexpr (kBoxes) {
          const bool out = g.x < ce.lb[0] || g.x > ce.ub[0] || g.y < ce.lb[1] || g.y > ce.ub[1] || g.z < ce.lb[2] ||
                           g.z > ce.ub[2];
          if (!wave_any(!out)) continue;
        }
        p = ce.prim;
        orig = ce.orig;
      }
      const DevPrim<float> Q = cload(vp, p);
      const float bound = bound_of(best + S.cfg);
      // every member sphere's value is at least the bounding centre's
      // distance minus the block's reach (the SDFs are 1-Lipschitz)
      if (!all && !wave_any(sdf_may_reach<K>(Q, g, bound + ereach))) continue;
      const uint32_t pkey = (uint32_t)orig * (uint32_t)ka.n_spheres;
      int cnt = 0;  // entries collected, wave-uniform
      auto flush = [&]() {
        wave_lds_order();
        if (S.lane < cnt) {
          const float* t = entries + S.lane;
          const V3<float> ec{t[0], t[64], t[128]};
          const float er = t[192];
          const float v = sdf_eval_kind<K>(Q, ec) - er;
          if (!outside_aabb(Q, ec, er + kCutoff)) offer(best + __float_as_int(t[320]), v, (uint32_t)__float_as_int(t[256]));
        }
        wave_lds_order();
        cnt = 0;
      };
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const bool pass = k < n && sdf_may_reach<K>(Q, c[k], bound + r[k]);
        const uint64_t m = __ballot(pass);
        if (m == 0) continue;
        const int more = __popcll(m);
        if (cnt + more > 64) flush();
        const uint32_t key = key_of(k);
        if (pass) {
          float* t = entries + cnt + lane_rank(m);
          t[0] = c[k].x;
          t[64] = c[k].y;
          t[128] = c[k].z;
          t[192] = r[k];
          t[256] = __int_as_float((int)(key + pkey));
          t[320] = __int_as_float(S.cfg);
        }
        cnt += more;
      }
      if (cnt > 0) flush();
    }
  };
  kind(std::integral_constant<int, kKindBoxAA>{});
  kind(std::integral_constant<int, kKindBoxRot>{});
  kind(std::integral_constant<int, kKindCylZ>{});
  kind(std::integral_constant<int, kKindCylRot>{});
  kind(std::integral_constant<int, kKindSphere>{});
  kind(std::integral_constant<int, kKindGround>{});
  // Clouds: sqrt(min |c - p|^2) - rc - r (CloudSDF::evaluate,
  // primitive_sdf.hpp:585-590, minus the sphere radius) after the reference's
  // AABB prefilter grown by the cutoff.  Only points within r + rc + cutoff of
  // a sphere can give a value below the cutoff, so the minimum is taken over
  // the tiles within that reach of the block (all tiles when the rotation is
  // outside the norm bounds).
  if (H < kCloudLanes || !it.first) return;
  for (int p = sc.vrange[kKindCloud]; p < sc.vrange[kKindCloud + 1]; ++p) {
    const DevPrim<float> Pc = cload(vp, p);
    const uint32_t pkey = (uint32_t)cload(sc.vorig, p) * (uint32_t)ka.n_spheres;
    const float rc = Pc.p0;
    const float reach = bk.G * bk.n2_hi + rc + kCutoff + 1e-5f;
    float d2[NK];
    cloud_block_min<NK>(sc, (Pc.flags >> 4) & 15, c, n, g, all ? FLT_MAX : reach * reach, true, d2);
#pragma unroll
    for (int k = 0; k < NK; ++k)
      if (k < n && d2[k] != FLT_MAX && !outside_aabb(Pc, c[k], r[k] + kCutoff))
        offer(best + S.cfg, sqrtf(d2[k]) - rc - r[k], key_of(k) + pkey);
  }
}

// One self pair; with H > 1 a configuration's lanes share its first group's
// spheres.
template <int H>
__device__ __forceinline__ void self_pair(const Stage<H>& S, const KinArgs<float>& ka, int k, Best* best) {
  const DevSelfPair pr = cload(ka.pairs, k);
  const Pose<float> P1 = S.pose(pr.pose1), P2 = S.pose(pr.pose2);
  const M3<float> R1 = qmat(P1.q), R2 = qmat(P2.q);
  // the groups' bounding spheres; |R v| <= grow |v| for a rotation matrix of a
  // quaternion with |q|^2 = n, grow = 1 + 2 |n - 1|.  A sphere pair's value is
  // at least the groups' distance minus their reach.
  const V3<float> g1 = add(mv(R1, V3<float>{pr.bound1[0], pr.bound1[1], pr.bound1[2]}), P1.t);
  const V3<float> g2 = add(mv(R2, V3<float>{pr.bound2[0], pr.bound2[1], pr.bound2[2]}), P2.t);
  const float n1 = P1.q.x * P1.q.x + P1.q.y * P1.q.y + P1.q.z * P1.q.z + P1.q.w * P1.q.w;
  const float n2 = P2.q.x * P2.q.x + P2.q.y * P2.q.y + P2.q.z * P2.q.z + P2.q.w * P2.q.w;
  const float dn = fmaxf(fabsf(n1 - 1.0f), fabsf(n2 - 1.0f));
  const float reach = (pr.bound1[3] + pr.bound2[3]) * (1.0f + 2.0f * dn);
  const V3<float> dg = sub(g1, g2);
  float bound = bound_of(best + S.cfg);
  if (!wave_any(!(sqrtf(dot(dg, dg)) - reach > bound + 1e-5f))) return;
  for (int i0 = pr.begin1; i0 < pr.end1; i0 += H) {
    const int i = H == 1 ? i0 : i0 + S.sub;
    const bool live = i < pr.end1;
    DevSphere<float> a{};
    if constexpr (H == 1)
      a = cload(ka.spheres, i);
    else if (live)
      a = ka.spheres[i];
    const V3<float> ci = add(mv(R1, V3<float>{a.x, a.y, a.z}), P1.t);
    for (int j = pr.begin2; j < pr.end2; ++j) {
      const DevSphere<float> bb = cload(ka.spheres, j);
      const V3<float> cj = add(mv(R2, V3<float>{bb.x, bb.y, bb.z}), P2.t);
      const V3<float> d = sub(ci, cj);
      const float d2 = dot(d, d), rs = a.r + bb.r;
      // may d - rs be below the bound?  (no correctly rounded root yet)
      const float L = fmaxf(bound + rs, 0.0f) + 1e-5f;
      if (live && !(d2 > L * L * 1.0001f)) {
        offer(best + S.cfg, sqrtf(d2) - rs,
              ((uint32_t)k << (2 * kSelfPosBits)) | ((uint32_t)(i - pr.begin1) << kSelfPosBits) |
                  (uint32_t)(j - pr.begin2));
        bound = bound_of(best + S.cfg);
      }
    }
  }
}

// Smoothness cost of one trajectory by a wave (smoothcost_fullmat,
// nlp_solver/sqp_based_solver.py:74-96):
//   cost = sum_{interior t} sum_j w_j^2 a_{t,j}^2,  a_t = x_{t-1} - 2 x_t + x_{t+1},
// terms and sums in FP64 (a fixed order), rounded once.
__device__ __forceinline__ void traj_cost(const StagedOut& o, const double* X, int64_t ldx, int D, int i, int lane) {
  const int64_t b0 = o.offsets[i], T = o.offsets[i + 1] - b0;
  double c = 0.0;
  for (int64_t t = 1 + lane; t + 1 < T; t += 64) {
    const double* x = X + b0 + t;
    for (int j = 0; j < D; ++j, x += ldx) {
      const double a = x[-1] - 2.0 * x[0] + x[1];
      c += o.w2[j] * a * a;
    }
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) c += __shfl_xor(c, s, 64);
  if (lane == 0) o.cost[i] = (float)c;
}

// Bound by latency: scalar table reads and LDS.  Measured: trajectories of the
// dual arm (123,498 waypoints) 411 -> 138 us, 8,192 configurations of the 7R arm
// among 32 primitives 51 -> 17 us, 256 among two bars 28 -> 12 us, each against
// a lane per configuration (a workgroup of 8 waves with a block each, every wave
// walking FK again) before.
// kShared: the robot's q columns drive several joints (ka.shared).
template <int H, bool kShared>
__device__ __forceinline__ void eval_staged(const KinArgs<float>& ka, const SceneArgs<float>& sc, const double* q,
                                            int64_t ldq, int64_t B, const StagedOut& o, const StageLds& lay) {
  HIP_DYNAMIC_SHARED(float, staged_lds)
  const Stage<H> S(staged_lds, lay);
  constexpr int C = Stage<H>::C;
  const int lane = S.lane, w = S.w, W = S.W, cfg = S.cfg, D = ka.n_cols, NP = sc.n_prims;
  if ((int)blockIdx.x >= o.n_chunks) {
    const int i = ((int)blockIdx.x - o.n_chunks) * W + w;
    if (i < o.n_traj) traj_cost(o, q, ldq, D, i, lane);
    return;
  }
  const int64_t b = (int64_t)blockIdx.x * C + cfg;
  const bool active = b < B;
  BatchQ qs{q, ldq, active ? b : B - 1};
  // scratch: what the candidates' compaction needs per wave, then the winners
  // (kWinWords each), over the joints' words, which only the walk reads; the
  // best external and self pair; waypoint within its trajectory and its
  // length; the queue
  float* scratch = staged_lds + o.scratch;
  float* win = scratch;
  Best* best = reinterpret_cast<Best*>(staged_lds + o.best);
  int* tr = reinterpret_cast<int*>(best + 2 * C);
  int* queue = tr + 2 * C;
  const int n_blocks = ka.n_units - ka.n_pairs;
  S.joints(ka, qs, false);
  if (threadIdx.x < 2 * C) best[threadIdx.x] = no_winner();
  if (threadIdx.x == 0) *queue = 0;
  __syncthreads();
  S.walk(ka, qs);
  if (w >= ka.n_paths) {
    const int part = w - ka.n_paths, parts = W - ka.n_paths;
    warm_scalar(sc.vprims, sc.n_prims * (int)sizeof(DevPrim<float>), part, parts);
    warm_scalar(ka.blocks, n_blocks * (int)sizeof(DevSphereBlock), part, parts);
    if (o.sliced) {
      warm_scalar(sc.ecull, sc.n_ecull * (int)sizeof(CullEntry), part, parts);
      warm_scalar(sc.eslices, sc.n_eslices * (int)sizeof(DevCullSlice), part, parts);
      warm_scalar(sc.ecull_range, n_blocks * (int)sizeof(CullRange), part, parts);
    }
  }
  if (o.offsets && w == W - 1 && S.sub == 0) {
    int lo = 0, hi = o.n_traj;  // offsets[lo] <= b < offsets[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (o.offsets[mid] <= qs.b) lo = mid;
      else hi = mid;
    }
    const int64_t b0 = o.offsets[lo];
    tr[cfg] = (int)(qs.b - b0);
    tr[C + cfg] = (int)(o.offsets[lo + 1] - b0);
  }
  __syncthreads();
  const int n_ext = NP == 0 ? 0 : (o.sliced ? sc.n_eslices : n_blocks);
  const int n_items = n_ext + ka.n_pairs;
  for (;;) {
    int it = 0;
    if (lane == 0) it = atomicAdd(queue, 1);
    it = __builtin_amdgcn_readfirstlane(it);
    if (it >= n_items) break;
    if (it < n_ext) {
      float* entries = scratch + w * 64 * kEntryWords;
      if (o.sliced) {
        ext_slice<H, false>(S, ka, sc, cload(sc.eslices, it), best, entries);
      } else {
        const CullRange cr = cload(sc.ecull_range, n_ext - 1 - it);
        ext_slice<H, true>(S, ka, sc, DevCullSlice{n_ext - 1 - it, cr.at[0], cr.at[kKindCloud], 1}, best, entries);
      }
    } else {
      self_pair<H>(S, ka, it - n_ext, best + C);
    }
  }
  __syncthreads();
  // The winners: waves 0 to 2 the external ones, by primitive type (so that no
  // wave runs more than one gradient's branches), wave 3 the self pairs; with
  // fewer waves, one after the other.
  auto put3 = [&](int at, V3<float> v) {
    win[at * C + cfg] = v.x;
    win[(at + 1) * C + cfg] = v.y;
    win[(at + 2) * C + cfg] = v.z;
  };
  auto put_mask = [&](int at, uint64_t m) {
    win[at * C + cfg] = __int_as_float((int)(uint32_t)m);
    win[(at + 1) * C + cfg] = __int_as_float((int)(uint32_t)(m >> 32));
  };
  auto centre = [&](int out, uint64_t& mask) {
    const DevSphereRow a = ka.rows[out];  // per-lane index: vector loads
    mask = a.col_mask;
    const Pose<float> P = S.pose(a.pose);
    return add(mv(qmat(P.q), V3<float>{a.x, a.y, a.z}), P.t);
  };
  for (int job = w; job < 4 && S.sub == 0; job += W) {
    if (job < 3 && NP > 0) {
      const Best e = best[cfg];
      if (!has_winner(e)) {
        if (job == 0) {
          put3(3, V3<float>{0.f, 0.f, 0.f});
          put_mask(6, 0);
          if (active) o.vals[b] = kCutoff;
        }
      } else {
        const uint32_t key = (uint32_t)e;
        const int out = (int)(key % (uint32_t)ka.n_spheres), orig = (int)(key / (uint32_t)ka.n_spheres % (uint32_t)NP);
        const DevPrim<float>& Q = reinterpret_cast<const DevPrim<float>*>(sc.prims)[orig];
        uint64_t m0;
        const V3<float> c0 = centre(out, m0);
        const int type = Q.type;
        if (job == (type == PMP_PRIM_BOX ? 0 : (type == PMP_PRIM_CYLINDER ? 1 : 2))) {
          V3<float> g0;
          if (type == PMP_PRIM_CLOUD) {
            // the gradient of sqrt(min |c - p|^2) at the nearest point, which the
            // reference's forward difference (eps 1e-6) approximates
            float d2;
            const V3<float> d = sub(c0, cloud_nearest(sc, (Q.flags >> 4) & 15, c0, d2));
            g0 = scale(1.0f / sqrtf(dot(d, d)), d);
          } else {
            g0 = sdf_grad(Q, c0);
          }
          put3(0, c0);
          put3(3, g0);
          put_mask(6, m0);
          if (active) o.vals[b] = best_value(e);
        }
      }
    }
    if (job == 3 && ka.n_pairs > 0) {
      const Best e = best[C + cfg];
      V3<float> n{0.f, 0.f, 0.f};
      uint64_t m1 = 0, m2 = 0;
      if (has_winner(e)) {
        const uint32_t key = (uint32_t)e, mask = (1u << kSelfPosBits) - 1;
        const DevSelfPair& pr = ka.pairs[key >> (2 * kSelfPosBits)];
        const V3<float> c1 = centre(ka.meta[pr.begin1 + (int)((key >> kSelfPosBits) & mask)].out, m1);
        const V3<float> c2 = centre(ka.meta[pr.begin2 + (int)(key & mask)].out, m2);
        const V3<float> d = sub(c1, c2);
        n = scale(1.0f / sqrtf(dot(d, d)), d);
        put3(8, c1);
        put3(11, c2);
      }
      put3(14, n);
      put_mask(17, m1);
      put_mask(19, m2);
      if (active) o.vals[(NP > 0 ? B : 0) + b] = best_value(e);
    }
  }
  __syncthreads();
  auto get3 = [&](int at) { return V3<float>{win[at * C + cfg], win[(at + 1) * C + cfg], win[(at + 2) * C + cfg]}; };
  auto get_bit = [&](int at, int j) { return (__float_as_int(win[(at + (j >> 5)) * C + cfg]) >> (j & 31)) & 1; };
  const int t = o.offsets ? tr[cfg] : 0, T = o.offsets ? tr[C + cfg] : 0;
  for (int j = w * H + S.sub; j < D; j += W * H) {
    const bool rev = (ka.rev_mask >> j) & 1ull;
    V3<float> a{0.f, 0.f, 0.f}, og{0.f, 0.f, 0.f};
    S.frame(ka, qs, j, a, og);
    auto col = [&](int at, V3<float> c) {
      if (!get_bit(at, j)) return V3<float>{0.f, 0.f, 0.f};
      return rev ? cross(a, sub(c, og)) : a;
    };
    // the winners' nodes again from their keys
    auto joints_col = [&](int node, V3<float> c) {
      V3<float> r{0.f, 0.f, 0.f};
      S.joint_columns(ka, node, c, [&](int at, V3<float> v) {
        if (at == j) r = add(r, v);
      });
      return r;
    };
    if (!active) continue;
    const bool by_joint = kShared && j < ka.n_q_cols;
    if (NP > 0) {
      if (by_joint) {
        const Best e = best[cfg];
        float v = 0.f;
        if (has_winner(e)) v = dot(get3(3), joints_col(ka.rows[(uint32_t)e % (uint32_t)ka.n_spheres].node, get3(0)));
        o.jac[(int64_t)j * B + b] = v;
      } else {
        o.jac[(int64_t)j * B + b] = dot(get3(3), col(6, get3(0)));
      }
    }
    if (ka.n_pairs > 0) {
      float* row = o.jac + ((NP > 0 ? (int64_t)D : 0) + j) * B + b;
      if (by_joint) {
        const Best e = best[C + cfg];
        float v = 0.f;
        if (has_winner(e)) {
          const DevSelfPair& pr = ka.pairs[(uint32_t)e >> (2 * kSelfPosBits)];
          v = dot(get3(14), sub(joints_col(pr.node1, get3(8)), joints_col(pr.node2, get3(11))));
        }
        *row = v;
      } else {
        *row = dot(get3(14), sub(col(17, get3(8)), col(19, get3(11))));
      }
    }
    if (o.offsets) {
      // smoothness gradient: d cost / d x_t = 2 w^2 (a_{t-1} - 2 a_t + a_{t+1}),
      // terms of interior indices only; the differences in FP64 (they cancel)
      const double* x = q + (int64_t)j * ldq + b;
      auto acc = [&](int s) { return x[s - 1] - 2.0 * x[s] + x[s + 1]; };
      double g = 0.0;
      if (t - 1 >= 1 && t - 1 <= T - 2) g += acc(-1);
      if (t >= 1 && t <= T - 2) g -= 2.0 * acc(0);
      if (t + 1 >= 1 && t + 1 <= T - 2) g += acc(1);
      o.grad[(int64_t)j * B + b] = (float)(2.0 * o.w2[j] * g);
    }
  }
}

template <int H>
__global__ void __launch_bounds__(1024) eval_staged_kernel(KinArgs<float> ka, SceneArgs<float> sc, const double* q,
                                                           int64_t ldq, int64_t B, StagedOut o, StageLds lay) {
  eval_staged<H, false>(ka, sc, q, ldq, B, o, lay);
}
template <int H>
__global__ void __launch_bounds__(1024) eval_shared_kernel(KinArgs<float> ka, SceneArgs<float> sc, const double* q,
                                                           int64_t ldq, int64_t B, StagedOut o, StageLds lay) {
  eval_staged<H, true>(ka, sc, q, ldq, B, o, lay);
}

bool launch_eval_staged(const KinArgs<float>& ka, const SceneArgs<float>& sc, const double* q, int64_t ldq, int64_t B,
                        const EvalArgs& e, hipStream_t st, hipError_t* err) {
  if (!ka.staged || (uint64_t)ka.n_spheres * ka.n_spheres * sc.n_prims >= 0xffffffffu) return false;
  int o_scratch = 0, o_best = 0;
  auto lds_of = [&](int H, int W) {
    const int C = 64 / H;
    const StageLds L = stage_lds(ka, C);
    // the joints' words again, if they are enough
    const int need = (W * kEntryWords * 64 > kWinWords * C ? W * kEntryWords * 64 : kWinWords * C);
    o_scratch = need <= L.poses ? 0 : L.end;
    o_best = (L.end + (o_scratch ? need : 0) + 1) & ~1;
    return sizeof(float) * (size_t)(o_best + 4 * C + 2 * C + 1);
  };
  StageShape sh = stage_shape(B, ka.n_units - ka.n_pairs);
  // a block's cloud is one wave's work: with four lanes a configuration more of
  // its tiles are too far for all of a wave's configurations (10,000 of the
  // Fetch-like robot against 20,000 points 2,277 us, 2,926 with one lane, 2,785
  // before the staged form; 100,000 of the 7R arm 744, 1,105 and 1,646)
  if (sc.n_cloud > 0 && sh.H < kCloudLanes) sh.H = kCloudLanes;
  while (sh.H < 8 && lds_of(sh.H, sh.W) > (size_t)ka.lds_limit) sh.H *= 2;
  if (ka.shared && sh.H > 1) sh.H = 8;
  if (2 * lds_of(sh.H, sh.W) > (size_t)ka.lds_limit && lds_of(sh.H, 16) <= (size_t)ka.lds_limit) sh.W = 16;
  const int64_t chunks = (B + 64 / sh.H - 1) / (64 / sh.H), n_traj = e.offsets ? e.n_traj : 0;
  const int H = sh.H, W = waves_of_launch(chunks + n_traj, sh.W);
  const size_t lds = lds_of(H, W);
  if (lds > (size_t)ka.lds_limit) return false;
  StagedOut o{};
  o.vals = e.vals;
  o.jac = e.jac;
  o.offsets = e.offsets;
  o.n_traj = (int)n_traj;
  o.w2 = e.w2;
  o.cost = e.cost;
  o.grad = e.grad;
  o.n_chunks = (int)chunks;
  // slices balance a workgroup's waves; a full GPU does better without their
  // repeated set-up (trajectories of the dual arm: 157 us by blocks, 182 by slices)
  o.sliced = e.whole_chunks > 0 ? (B + 63) / 64 < e.whole_chunks : B <= 64 * kCus;
  const StageLds lay = stage_lds(ka, 64 / H);
  o.scratch = o_scratch;
  o.best = o_best;
  const dim3 grid((unsigned)(chunks + (o.n_traj + W - 1) / W)), block(64 * W);
  *err = hipSuccess;
  if (grid.x > 0) {
#define PMP_EVAL(H) *err = launch_last(eval_staged_kernel<H>, grid, block, lds, st, ka, sc, q, ldq, B, o, lay)
    if (ka.shared)
      *err = launch_last(H == 1 ? eval_shared_kernel<1> : eval_shared_kernel<8>, grid, block, lds, st, ka, sc, q, ldq,
                         B, o, lay);
    else if (H == 1)
      PMP_EVAL(1);
    else if (H == 2)
      PMP_EVAL(2);
    else if (H == 4)
      PMP_EVAL(4);
    else
      PMP_EVAL(8);
#undef PMP_EVAL
  }
  return true;
}

}  // namespace pmp
