// Signed distance of every (sphere, primitive) pair with its derivative, by
// staged workgroups (stage.hpp).  FK runs once per workgroup; a wave takes up
// to eight spheres of one link (distances) or one sphere (gradients) and a
// slice of the primitives, so everything a primitive's evaluation reads is
// wave-uniform.  Bound by the stores (a gradient batch writes S x P x (D + 1)
// floats per configuration); the evaluation is resolved per primitive kind,
// value and gradient together, to stay below that.
#include <algorithm>
#include <type_traits>

#include "last_launch.hpp"
#include "stage.hpp"

namespace pmp {

// Runs f with the primitive's kind as a compile-time constant (clouds excluded).
template <class F>
__device__ __forceinline__ void with_kind(const DevPrim<float>& p, F&& f) {
  // The empty statements keep the compiler from merging the cases' last stores
  // behind the switch (8,191 configurations' distances 27.7 us, 28.4 merged).
  switch (prim_kind(p)) {
    case kKindBoxAA:
      f(std::integral_constant<int, kKindBoxAA>{});
      asm volatile("; box");
      break;
    case kKindBoxRot:
      f(std::integral_constant<int, kKindBoxRot>{});
      asm volatile("; rotated box");
      break;
    case kKindCylZ:
      f(std::integral_constant<int, kKindCylZ>{});
      asm volatile("; cylinder");
      break;
    case kKindCylRot:
      f(std::integral_constant<int, kKindCylRot>{});
      asm volatile("; rotated cylinder");
      break;
    case kKindSphere:
      f(std::integral_constant<int, kKindSphere>{});
      asm volatile("; sphere");
      break;
    default:
      f(std::integral_constant<int, kKindGround>{});
      asm volatile("; ground");
  }
}
// CloudSDF::evaluate (primitive_sdf.hpp:585-590): sqrt of the nearest squared
// distance minus r_cloud; its gradient at the nearest point.
__device__ __forceinline__ float cloud_eval(const SceneArgs<float>& sc, const DevPrim<float>& P, V3<float> c,
                                            V3<float>& g) {
  float d2;
  const V3<float> dv = sub(c, cloud_nearest<true>(sc, (P.flags >> 4) & 15, c, d2));
  g = scale(1.0f / sqrtf(dot3(dv, dv)), dv);
  return sqrtf(d2) - P.p0;
}

// The joint frames of every column, [D][6][C] from `at`, by all waves after
// the walk.
template <int H, class QS>
__device__ __forceinline__ float* stage_frames(const Stage<H>& S, const KinArgs<float>& ka, const QS& qs, int at) {
  constexpr int C = Stage<H>::C;
  float* frames = S.lds + at;
  for (int j = S.w * H + S.sub; j < ka.n_cols; j += S.W * H) {
    V3<float> a{0.f, 0.f, 0.f}, o{0.f, 0.f, 0.f};
    S.frame(ka, qs, j, a, o);
    float* f = frames + 6 * j * C + S.cfg;
    f[0] = a.x;
    f[C] = a.y;
    f[2 * C] = a.z;
    f[3 * C] = o.x;
    f[4 * C] = o.y;
    f[5 * C] = o.z;
  }
  return frames;
}
template <int C>
__device__ __forceinline__ void staged_frame(const float* frames, int j, int cfg, V3<float>& a, V3<float>& o) {
  const float* f = frames + 6 * j * C + cfg;
  a = {f[0], f[C], f[2 * C]};
  o = {f[3 * C], f[4 * C], f[5 * C]};
}

// The (share, chunk of 64 configurations) of a workgroup: workgroups go to the
// XCDs in turn, and each XCD gets a contiguous range, chunk fastest, so that
// the chunks that write the same rows (and, in rows that do not start on a
// cache line, the same lines) share an L2.
__device__ __forceinline__ void share_and_chunk(int chunks, int& share, int& chunk) {
  const int g = (int)blockIdx.x, n = (int)gridDim.x, x = g % kXcds;
  const int at = x * (n / kXcds) + min(x, n % kXcds) + g / kXcds;
  share = at / chunks;
  chunk = at % chunks;
}

// Rows that start on a cache line are written once and in whole lines:
// streaming stores keep them from displacing one another in L2.  Lines shared
// by two waves are left to L2 to complete.
template <bool kStream>
__device__ __forceinline__ void put(float* p, float v) {
  if constexpr (kStream)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// dist[(s * P + p) * B + b]: task t of the launch is item t / n_slices (up to
// eight spheres of a link, so that a primitive is read once for all of them)
// against slice t % n_slices of the primitives; workgroups share the tasks.
template <int H, bool kStream>
__global__ void __launch_bounds__(512) pair_dist_kernel(KinArgs<float> ka, SceneArgs<float> sc, const double* q,
                                                        int64_t ldq, int64_t B, float* dist, int n_slices, int chunks,
                                                        StageLds lay) {
  HIP_DYNAMIC_SHARED(float, staged_lds)
  const Stage<H> S(staged_lds, lay);
  int share, chunk;
  share_and_chunk(chunks, share, chunk);
  const int shares = (int)gridDim.x / chunks;
  const int64_t b = (int64_t)chunk * Stage<H>::C + S.cfg;
  const bool active = b < B && S.sub == 0;
  BatchQ qs{q, ldq, b < B ? b : B - 1};
  // coordinates beyond the forms of sdf_value_grad: looked for by the waves that
  // have nothing to walk
  int* flag = reinterpret_cast<int*>(S.lds + lay.end);
  if (threadIdx.x == 0) *flag = ka.far | sc.far;
  S.joints(ka, qs, false);
  __syncthreads();
  S.walk(ka, qs);
  const int idle = ka.n_paths < S.W ? ka.n_paths : 0;  // the first such wave
  bool any_far = false;
  if (S.w >= idle)
    for (int col = (S.w - idle) * H + S.sub; col < ka.n_cols; col += (S.W - idle) * H)
      any_far = any_far || !(fabs(qs.get(col)) < 0.1 * kFar);
  if (any_far) *flag = 1;
  if (S.w >= ka.n_paths)
    warm_scalar(sc.prims, sc.n_prims * (int)sizeof(DevPrim<float>), S.w - ka.n_paths, S.W - ka.n_paths);
  __syncthreads();
  const bool far = __builtin_amdgcn_readfirstlane(*flag) != 0;
  const int NP = sc.n_prims, T = ka.n_items * n_slices, t_end = (int)((int64_t)T * (share + 1) / shares);
  int t = (int)((int64_t)T * share / shares) + S.w;
  for (; far && t < t_end; t += S.W) {
    const DevSphereItem it = cload(ka.items, t / n_slices);
    const int sl = t % n_slices, p_end = (int)((int64_t)NP * (sl + 1) / n_slices);
    const Pose<float> P = S.pose(it.pose);
    for (int s = it.begin; s < it.end; ++s) {
      const DevSphere<float> a = cload(ka.spheres, s);
      const V3<float> c = add(mv3(qmat(P.q), V3<float>{a.x, a.y, a.z}), P.t);
      float* row = dist + (int64_t)cload(ka.meta, s).out * NP * B + b;
      for (int p = (int)((int64_t)NP * sl / n_slices); p < p_end; ++p) {
        const float d = sdf_eval(prim_at(sc, p), c) - a.r;
        if (active) put<kStream>(row + (int64_t)p * B, d);
      }
    }
  }
  for (; t < t_end; t += S.W) {
    const DevSphereItem it = cload(ka.items, t / n_slices);
    const int sl = t % n_slices, n = it.end - it.begin;
    const Pose<float> P = S.pose(it.pose);
    const M3<float> R = qmat(P.q);
    V3<float> c[kItemSpheres];
    float r[kItemSpheres];
    float* row[kItemSpheres];
#pragma unroll
    for (int k = 0; k < kItemSpheres; ++k) {
      const int s = min(it.begin + k, it.end - 1);
      const DevSphere<float> a = cload(ka.spheres, s);
      c[k] = add(mv3(R, V3<float>{a.x, a.y, a.z}), P.t);
      r[k] = a.r;
      row[k] = dist + (int64_t)cload(ka.meta, s).out * NP * B;
    }
    const int p_begin = (int)((int64_t)NP * sl / n_slices), p_end = (int)((int64_t)NP * (sl + 1) / n_slices);
    for (int p = p_begin; p < p_end; ++p) {
      const DevPrim<float> Q = prim_at(sc, p);
      with_kind(Q, [&](auto kc) {
#pragma unroll
        for (int k = 0; k < kItemSpheres; ++k) {
          if (k < n) {
            float d;
            V3<float> g;
            sdf_value_grad<decltype(kc)::value, false>(Q, c[k], d, g);
            if (active) put<kStream>(row[k] + (int64_t)p * B + b, d - r[k]);
          }
        }
      });
    }
  }
}

// dist as above and grad[((s * P + p) * D + j) * B + b]: task t is sphere
// t / n_slices (group order) against a slice of the primitives, MAXC columns
// at a time.  Bound by its stores: 8,192 configurations of the 7R arm against
// 32 primitives write 504 MB in 100 us (124 us with a lane per (configuration,
// link) before); 256-byte pieces of rows alone take 94 us on this card, a
// plain fill 73 us.  With rows off the cache lines (8,191 configurations) 142
// us; 277 us with streaming stores and neighbouring chunks on different XCDs.
// kShared: the robot's q columns drive several joints (ka.shared).
// kCloud: the scene holds clouds.  Finding the nearest point costs more than all
// else, so it is done once a sphere, before the columns, and distances alone
// (grad == nullptr) come here too, a sphere a task.  (2,000 configurations
// against 20,000 points: 31 joints, a search for every 16 of 37 columns 6,579 us,
// now 1,036, 3,027 before the staged form; 60 joints 28,221, 3,315 and 3,420;
// distances of the 7R arm, eight spheres a task 1,250, now 202, before 1,301.)
template <int H, int MAXC, bool kStream, bool kShared, bool kCloud>
__device__ __forceinline__ void pair_grad(const KinArgs<float>& ka, const SceneArgs<float>& sc, const double* q,
                                          int64_t ldq, int64_t B, float* dist, float* grad, int n_slices, int chunks,
                                          const StageLds& lay) {
  HIP_DYNAMIC_SHARED(float, staged_lds)
  const Stage<H> S(staged_lds, lay);
  int share, chunk;
  share_and_chunk(chunks, share, chunk);
  const int shares = (int)gridDim.x / chunks, cfg = S.cfg;
  const int64_t b = (int64_t)chunk * Stage<H>::C + cfg;
  const bool active = b < B && S.sub == 0;
  BatchQ qs{q, ldq, b < B ? b : B - 1};
  const int D = kCloud && !grad ? 0 : ka.n_cols;
  S.joints(ka, qs, false);
  __syncthreads();
  S.walk(ka, qs);
  __syncthreads();
  const int NP = sc.n_prims, T = ka.n_spheres * n_slices;
  const float* frames = nullptr;
  if (!kCloud || grad) {
    frames = stage_frames(S, ka, qs, lay.end);
    __syncthreads();
  }
  const int t_end = (int)((int64_t)T * (share + 1) / shares);
  for (int t = (int)((int64_t)T * share / shares) + S.w; t < t_end; t += S.W) {
    const int s = t / n_slices, sl = t % n_slices;
    const DevSphereRow row = cload(ka.rows, s);
    const Pose<float> P = S.pose(row.pose);
    const V3<float> c = add(mv3(qmat(P.q), V3<float>{row.x, row.y, row.z}), P.t);
    const int p_begin = (int)((int64_t)NP * sl / n_slices), p_end = (int)((int64_t)NP * (sl + 1) / n_slices);
    V3<float> near[kMaxClouds];
    if constexpr (kCloud) {
      for (int p = p_begin; p < p_end; ++p) {
        const DevPrim<float> Q = prim_at(sc, p);
        if (Q.type != PMP_PRIM_CLOUD) continue;
        V3<float> g;
        const float d = cloud_eval(sc, Q, c, g);
#pragma unroll
        for (int k = 0; k < kMaxClouds; ++k)
          if (k == ((Q.flags >> 4) & 15)) near[k] = g;
        if (active) put<kStream>(dist + ((int64_t)s * NP + p) * B + b, d - row.r);
      }
    }
    for (int j0 = 0; j0 < D || j0 == 0; j0 += MAXC) {
      V3<float> J[MAXC];
#pragma unroll
      for (int j = 0; j < MAXC; ++j) {
        J[j] = {0.f, 0.f, 0.f};
        if (j0 + j < D && ((row.col_mask >> (j0 + j)) & 1ull)) {
          V3<float> a, o;
          staged_frame<Stage<H>::C>(frames, j0 + j, cfg, a, o);
          J[j] = ((ka.rev_mask >> (j0 + j)) & 1ull) ? cross(a, sub(c, o)) : a;
          if (kShared && j0 + j < ka.n_q_cols) J[j] = {0.f, 0.f, 0.f};
        }
      }
      if constexpr (kShared)
        S.joint_columns(ka, row.node, c, [&](int col, V3<float> v) {
#pragma unroll
          for (int j = 0; j < MAXC; ++j)
            if (j0 + j == col) J[j] = add(J[j], v);
        });
      for (int p = p_begin; p < p_end; ++p) {
        const DevPrim<float> Q = prim_at(sc, p);
        float d = 0.f;
        V3<float> g{0.f, 0.f, 0.f};
        const bool cloud = kCloud && Q.type == PMP_PRIM_CLOUD;
        if (cloud) {
#pragma unroll
          for (int k = 0; k < kMaxClouds; ++k)
            if (k == ((Q.flags >> 4) & 15)) g = near[k];
        } else {
          with_kind(Q, [&](auto kc) { sdf_value_grad<decltype(kc)::value, true>(Q, c, d, g); });
        }
        if (!active) continue;
        const int64_t at = (int64_t)s * NP + p;
        if (j0 == 0 && !cloud) put<kStream>(dist + at * B + b, d - row.r);
        float* gp = grad + (at * D + j0) * B + b;
#pragma unroll
        for (int j = 0; j < MAXC; ++j) {
          if (j0 + j < D) {
            put<kStream>(gp, dot3(g, J[j]));
            gp += B;
          }
        }
      }
    }
  }
}

template <int H, int MAXC, bool kStream>
__global__ void __launch_bounds__(256) pair_grad_kernel(KinArgs<float> ka, SceneArgs<float> sc, const double* q,
                                                        int64_t ldq, int64_t B, float* dist, float* grad, int n_slices,
                                                        int chunks, StageLds lay) {
  pair_grad<H, MAXC, kStream, false, false>(ka, sc, q, ldq, B, dist, grad, n_slices, chunks, lay);
}
template <int H>
__global__ void __launch_bounds__(256) pair_grad_shared_kernel(KinArgs<float> ka, SceneArgs<float> sc, const double* q,
                                                               int64_t ldq, int64_t B, float* dist, float* grad,
                                                               int n_slices, int chunks, StageLds lay) {
  pair_grad<H, 16, false, true, false>(ka, sc, q, ldq, B, dist, grad, n_slices, chunks, lay);
}
template <int H>
__global__ void __launch_bounds__(1024) pair_cloud_kernel(KinArgs<float> ka, SceneArgs<float> sc, const double* q,
                                                          int64_t ldq, int64_t B, float* dist, float* grad,
                                                          int n_slices, int chunks, StageLds lay) {
  pair_grad<H, 16, false, false, true>(ka, sc, q, ldq, B, dist, grad, n_slices, chunks, lay);
}
template <int H>
__global__ void __launch_bounds__(1024) pair_cloud_shared_kernel(KinArgs<float> ka, SceneArgs<float> sc,
                                                                 const double* q, int64_t ldq, int64_t B, float* dist,
                                                                 float* grad, int n_slices, int chunks, StageLds lay) {
  pair_grad<H, 16, false, true, true>(ka, sc, q, ldq, B, dist, grad, n_slices, chunks, lay);
}

constexpr int64_t kPairWorkgroups = 16 * kCus;

hipError_t launch_pairs(const KinArgs<float>& ka, const SceneArgs<float>& sc, const double* q, int64_t ldq,
                        int64_t B, float* dist, float* grad, int shares, hipStream_t st) {
  if (ka.n_spheres == 0 || sc.n_prims == 0 || B == 0) return hipSuccess;
  // 64 configurations a workgroup; robots whose tables do not fit take fewer
  // (H lanes hold a configuration, one of them works)
  int H = 1;
  auto lds_of = [&](int H) {
    return sizeof(float) * (size_t)(stage_lds(ka, 64 / H).end + (grad ? 6 * ka.n_cols * (64 / H) : 1));
  };
  while (H < 8 && lds_of(H) > (size_t)ka.lds_limit) H *= 2;
  if (grad && ka.shared && H > 1) H = 8;
  const size_t lds = lds_of(H);
  if (lds > (size_t)ka.lds_limit) return hipErrorInvalidConfiguration;  // 8 configurations of any robot fit
  const StageLds lay = stage_lds(ka, 64 / H);
  const int64_t chunks = (B + 64 / H - 1) / (64 / H);
  // With clouds a task a wave, of more primitives once there are waves enough
  // (those of a slice without a cloud end at once), four waves a workgroup while
  // that gives every CU one at most, and later as many as make 16 on a CU.
  // Distances: 4 primitives a task and a task a wave (8,191 configurations of
  // the 7R arm, 32 primitives: 31 us; 8 primitives 33, 4 tasks a wave 35).
  // Gradients: 8 primitives, two tasks a wave once the launch fills the GPU
  // (8,192: 100 us, 4 primitives 106, four tasks 106), else one (1,000: 24 us,
  // two 28).  More than kPairWorkgroups workgroups only repeat the walk.
  const bool cloud = sc.n_cloud > 0, by_sphere = grad || cloud;
  const size_t fit = (size_t)ka.lds_limit / lds;
  const int per = cloud && chunks * ka.n_spheres > 4 * kCus ? 32 : (by_sphere ? 8 : 4);
  const int tasks_per_wave = grad && !cloud && chunks > 32 ? 2 : 1;
  const int n_slices = (sc.n_prims + per - 1) / per;
  const int64_t tasks = (int64_t)(by_sphere ? ka.n_spheres : ka.n_items) * n_slices;
  const int few = chunks * ((tasks + 3) / 4) <= kCus || fit >= 4 ? 4 : (fit >= 2 ? 8 : 16);
  const int W = waves_of_launch(chunks, cloud ? few : (grad ? 4 : 8));
  int64_t ny = std::min((tasks + tasks_per_wave * W - 1) / (tasks_per_wave * W),
                        (kPairWorkgroups + chunks - 1) / chunks);
  if (shares > 0) ny = std::min<int64_t>(shares, tasks);
  const bool stream = B % 32 == 0;
  const dim3 grid((unsigned)(chunks * ny)), block(64 * W);
#define PMP_DIST(H, STREAM)                                                                                           \
  launch_last(pair_dist_kernel<H, STREAM>, grid, block, lds, st, ka, sc, q, ldq, B, dist, n_slices, (int)chunks, lay)
#define PMP_GRAD(H, MAXC, STREAM)                                                                                     \
  launch_last(pair_grad_kernel<H, MAXC, STREAM>, grid, block, lds, st, ka, sc, q, ldq, B, dist, grad, n_slices,       \
              (int)chunks, lay)
#define PMP_CLOUD(KERNEL) \
  launch_last(KERNEL, grid, block, lds, st, ka, sc, q, ldq, B, dist, grad, n_slices, (int)chunks, lay)
  if (cloud && grad && ka.shared) return PMP_CLOUD((H == 1 ? pair_cloud_shared_kernel<1> : pair_cloud_shared_kernel<8>));
  if (cloud)
    return PMP_CLOUD((H == 1 ? pair_cloud_kernel<1> : H == 2 ? pair_cloud_kernel<2> : H == 4 ? pair_cloud_kernel<4>
                                                                                             : pair_cloud_kernel<8>));
#undef PMP_CLOUD
  if (grad && ka.shared)
    return launch_last(H == 1 ? pair_grad_shared_kernel<1> : pair_grad_shared_kernel<8>, grid, block, lds, st, ka, sc,
                       q, ldq, B, dist, grad, n_slices, (int)chunks, lay);
  if (H == 2) return grad ? PMP_GRAD(2, 16, false) : PMP_DIST(2, false);
  if (H == 4) return grad ? PMP_GRAD(4, 16, false) : PMP_DIST(4, false);
  if (H == 8) return grad ? PMP_GRAD(8, 16, false) : PMP_DIST(8, false);
  if (!grad) return stream ? PMP_DIST(1, true) : PMP_DIST(1, false);
  if (ka.n_cols <= 8) return stream ? PMP_GRAD(1, 8, true) : PMP_GRAD(1, 8, false);
  return stream ? PMP_GRAD(1, 16, true) : PMP_GRAD(1, 16, false);
#undef PMP_DIST
#undef PMP_GRAD
}

}  // namespace pmp
