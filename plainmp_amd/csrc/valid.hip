// Validity of a batch of configurations by staged workgroups (stage.hpp,
// valid_stage.hpp): SphereCollisionCst::is_valid_dirty
// (constraints/primitive_sphere_collision.cpp:181-254) per configuration.
#include "last_launch.hpp"
#include "valid_stage.hpp"

namespace pmp {

struct ValidOut {
  uint8_t* valid;
  int32_t* n_recheck;
  float band;
  int flags;  // LDS offset (floats)
  int whole_waves;
  bool sliced;
};

struct ValidKernelArgs {
  KinArgs<float> ka;
  SceneArgs<float> sc;
  KinArgs<double> k64;
  SceneArgs<double> s64;
  const double* q;
  int64_t ldq, B;
  ValidOut o;
  StageLds lay;
};

// Configurations left to FP64 whole, from arguments read again: the others'
// path keeps its registers.  (Out of line, 2.5 times the time.)
template <int H>
__device__ __forceinline__ void valid_whole(const Stage<H>& S, const ValidLds<false>& out) {
  const ValidKernelArgs& A = args_again<ValidKernelArgs>();
  const int64_t b0 = (int64_t)blockIdx.x * Stage<H>::C;
  decide_whole(S.lane, S.cfg, S.sub, Stage<H>::NK, S.w, A.o.whole_waves, A.k64, A.s64, A.ka.base_type == PMP_BASE_FIXED,
               b0 + S.cfg < A.B, out, [&](int i) { return BatchQ{A.q, A.ldq, min(b0 + i, A.B - 1)}; });
}

// Bound by latency, like evaluate.  Against a launch with a lane per
// configuration or per (configuration, block) and a second one re-deciding
// whole configurations in FP64: 100,003 configurations of the Fetch-like robot
// 263 -> 89 us (128 us of it the FP64 walks), 1,024 of the 7R arm 15.0 -> 9 us;
// 16,384 configurations against a 65,536-point cloud 92 -> 34 us (queries through
// memory, 98,304 waves and four launches before).
// kCloud: the scene holds clouds (their code costs the others registers: 4 % of
// the time of the 100,003).
template <int H, bool kCloud>
__global__ void __launch_bounds__(1024) valid_staged_kernel(ValidKernelArgs args) {
  HIP_DYNAMIC_SHARED(float, staged_lds)
  const KinArgs<float>& ka = args.ka;
  const SceneArgs<float>& sc = args.sc;
  const StageLds& lay = args.lay;
  const ValidOut& o = args.o;
  const double* q = args.q;
  const int64_t ldq = args.ldq, B = args.B;
  const Stage<H> S(staged_lds, lay);
  constexpr int C = Stage<H>::C;
  const int lane = S.lane, w = S.w, W = S.W, cfg = S.cfg;
  const int64_t b = (int64_t)blockIdx.x * C + cfg;
  const bool active = b < B;
  BatchQ qs{q, ldq, active ? b : B - 1};
  const bool taylor = ka.base_type == PMP_BASE_FIXED;  // constraints/primitive.hpp:59-61
  ValidLds<false> out{};
  out.flags = reinterpret_cast<int*>(staged_lds + o.flags);
  out.count = out.flags + C;
  int* queue = out.count + 1;
  out.pend = queue + 1;
  const int n_blocks = ka.n_units - ka.n_pairs;
  if (threadIdx.x < C) out.flags[threadIdx.x] = active ? 0 : kHit;  // past the batch: nothing to do
  if (threadIdx.x == 0) *out.count = *queue = 0;
  S.joints(ka, qs, taylor);
  __syncthreads();
  // joint values outside the FP32 walk's ranges
  for (int col = w * H + S.sub; col < ka.n_cols; col += W * H)
    if (!fp32_range_col(ka.rev_mask, col, qs.get(col))) out.mark(cfg, kWhole);
  S.walk(ka, qs);
  if (w >= ka.n_paths) {
    const int part = w - ka.n_paths, parts = W - ka.n_paths;
    warm_scalar(sc.vprims, sc.n_prims * (int)sizeof(DevPrim<float>), part, parts);
    warm_scalar(ka.blocks, n_blocks * (int)sizeof(DevSphereBlock), part, parts);
    warm_scalar(sc.cull, sc.n_cull * (int)sizeof(CullEntry), part, parts);
  }
  __syncthreads();
  valid_items<kCloud>(S, ka, sc, o.band, out, queue, kCloud || o.sliced);
  __syncthreads();
  const bool whole = any_whole(out, cfg);
  if (w == 0)
    decide_pending(lane, cfg, ka, args.k64, args.s64, taylor, out,
                   [&](int i) { return BatchQ{q, ldq, min((int64_t)blockIdx.x * C + i, B - 1)}; });
  if (whole) {
    __syncthreads();
    valid_whole(S, out);
    __syncthreads();
  }
  if (w != 0) return;
  const int f = out.state(cfg);
  if (active && S.sub == 0) {
    o.valid[b] = (f & kHit) ? 0 : 1;
    if (o.n_recheck && (f & kPended)) atomicAdd(o.n_recheck, 1);
  }
}

hipError_t launch_valid(const KinArgs<float>& k32, const KinArgs<double>& k64, const SceneArgs<float>& s32,
                        const SceneArgs<double>& s64, const double* q, int64_t ldq, int64_t B, float band,
                        uint8_t* valid, int32_t* n_recheck, int, const CloudWork&, const CloudRange*, int, int32_t*,
                        int32_t*, hipStream_t st) {
  ValidOut o{valid, n_recheck, band, 0, 1, true};
  auto lds_of = [&](int H) {
    const int C = 64 / H;
    const StageLds L = stage_lds(k32, C);
    o.flags = L.end;
    const int keep = k64.slot_wave_bytes / (int)sizeof(float);  // one wave's FP64 kept poses
    if (o.flags < keep) o.flags = keep;
    return sizeof(float) * (size_t)(o.flags + C + 2 + 3 * kPendMax);
  };
  StageShape sh = stage_shape(B, k32.n_units - k32.n_pairs);
  while (sh.H < 8 && lds_of(sh.H) > (size_t)k32.lds_limit) sh.H *= 2;
  if (2 * lds_of(sh.H) > (size_t)k32.lds_limit) sh.W = 16;
  sh.W = waves_of_launch((B + 64 / sh.H - 1) / (64 / sh.H), sh.W);
  o.sliced = slice_blocks(k32, sh.W);
  const size_t lds = lds_of(sh.H);
  if (lds > (size_t)k32.lds_limit) return hipErrorInvalidConfiguration;  // 8 configurations of any robot fit
  o.whole_waves = whole_waves(k64, sizeof(float) * (size_t)o.flags, sh.W);
  const int C = 64 / sh.H;
  const StageLds lay = stage_lds(k32, C);
  const dim3 grid((unsigned)((B + C - 1) / C)), block(64 * sh.W);
#define PMP_VALID(H) \
  launch_last(s32.n_cloud > 0 ? valid_staged_kernel<H, true> : valid_staged_kernel<H, false>, grid, block, lds, st, \
              ValidKernelArgs{k32, s32, k64, s64, q, ldq, B, o, lay})
  return sh.H == 1 ? PMP_VALID(1) : sh.H == 2 ? PMP_VALID(2) : sh.H == 4 ? PMP_VALID(4) : PMP_VALID(8);
#undef PMP_VALID
}

}  // namespace pmp
