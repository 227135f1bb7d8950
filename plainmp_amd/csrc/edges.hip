// The motion check by staged workgroups (stage.hpp, valid_stage.hpp): a
// workgroup per motion walks its states in the validator's visiting order, 64
// at a time, and stops at the first chunk that holds a colliding one
// (ompl/motion_validator.cpp:44-126).  The answer does not depend on the
// visiting order (every state must be valid); the farthest-first order only
// makes the first chunk the most informative.  A chunk of at most 32, 16 or 8
// states gives each of them 2, 4 or 8 lanes, which share a block's spheres.
//
// Bound by the latency of a motion's chain (endpoints, step ratio, states,
// FK, tests).  Against a wave per motion that walks its states alone: 64
// motions of the 7R arm a tenth of the joint range long 42 -> 17 us, 1,024 of
// the 14-joint robot across the range 211 -> 101 us; 4,096 motions against a
// 65,536-point cloud 1,036 -> 583 us (2,600 before when a state fell in the
// band and its FP64 test walked every tile).
#include <limits.h>

#include "last_launch.hpp"
#include "valid_stage.hpp"

namespace pmp {

// A motion needing more states than this (a step ratio below 2^-24) is
// reported invalid with n_checked = -1.
constexpr double kMaxEdgeStates = 16777216.0;

// LDS offsets (floats), and the lanes a state gets at least (robots whose
// tables do not fit 64 states).
struct EdgeLds {
  int flags, h_min;
};

// State t of the way between the endpoints, which are staged as [2][D].
struct StagedEdgeQ {
  const double* ends;
  int D;
  double t;
  bool at_end;
  __device__ __forceinline__ double get(int col) const {
    const double a = ends[col], b = ends[D + col];
    return at_end ? b : a + (b - a) * t;
  }
};

// Step ratio (ompl/motion_validator.cpp:89-126), FP64: lane i < D holds column
// i of the endpoints and widths.
__device__ __forceinline__ double edge_step_ratio(const EdgeArgs& ea, int D, double a, double b, double width,
                                                  double inv_width) {
  if (ea.vtype == PMP_VALIDATOR_BOX) {
    const double diff = b - a, asd = fabs(diff) * inv_width;
    double max_diff = -INFINITY;
    int longest = 0;
    for (int i = 0; i < D; ++i) {
      const double v = readlane64(asd, i);
      if (v > max_diff) {
        max_diff = v;
        longest = i;
      }
    }
    longest = __builtin_amdgcn_readfirstlane(longest);
    const double diff_longest = fabs(max_diff > -INFINITY ? readlane64(diff, longest) : 0.0);
    return diff_longest < 1e-6 ? INFINITY : readlane64(width, longest) / diff_longest;
  }
  const double diff = a - b;
  double d2 = 0.0;
  for (int i = 0; i < D; ++i) {
    const double v = readlane64(diff, i);
    d2 += v * v;
  }
  return ea.resolution / sqrt(d2);
}

// A motion's sequence of states: k = 0 is its end itself, k >= 1 is interior
// position k + 1 of the farthest-first sequence when n_test <= 128 and
// position k of the linear sweep otherwise (ompl/motion_validator.cpp:44-78).
struct EdgeStates {
  const double* ends;
  int D, n_wp;  // n_wp = n_test - 1 states
  double ratio;
  __device__ __forceinline__ StagedEdgeQ at(const EdgeArgs& ea, int k) const {
    double t = 0.0;
    if (k > 0) t = n_wp < 128 ? (double)ea.seq[n_wp * 128 + (k + 1)] * ratio : (double)k * ratio;
    return {ends, D, t, k == 0};
  }
};

struct EdgeKernelArgs {
  KinArgs<float> ka;
  SceneArgs<float> sc;
  KinArgs<double> k64;
  SceneArgs<double> s64;
  EdgeArgs ea;
  EdgeLds el;
  float band;
};

// The FP32 items of states [base, base + 64 / H) of a motion.  Every thread
// takes part; the results are complete on return.
template <bool kCloud, int H>
__device__ __forceinline__ void edge_chunk(float* lds, const EdgeStates& es, int base, const ValidLds<true>& out,
                                           int* queue) {
  const EdgeKernelArgs& A = args_again<EdgeKernelArgs>();
  const KinArgs<float>& ka = A.ka;
  const SceneArgs<float>& sc = A.sc;
  const bool taylor = ka.base_type == PMP_BASE_FIXED;  // constraints/primitive.hpp:59-61
  constexpr int C = 64 / H;
  const StageLds lay = stage_lds(ka, C);
  const Stage<H> S(lds, lay);
  const int lane = S.lane, w = S.w, W = S.W, cfg = S.cfg;
  const bool active = base + cfg < es.n_wp;
  const StagedEdgeQ qs = es.at(A.ea, active ? base + cfg : 0);
  const int n_blocks = ka.n_units - ka.n_pairs;
  if (threadIdx.x < C) out.flags[threadIdx.x] = active ? 0 : kHit;  // past the motion: nothing to do
  if (threadIdx.x == 0) {
    *out.count = *queue = 0;
    *out.first = INT_MAX;
  }
  S.joints(ka, qs, taylor);
  __syncthreads();
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
  // whole blocks, or with clouds slices (of the solids beside them): a choice at
  // run time spills 20 to 50 more registers (against a cloud 583 -> 830 us)
  valid_items<kCloud>(S, ka, sc, A.band, out, queue, kCloud);
  __syncthreads();
}

// The FP64 decisions of a chunk, by the first wave: whether there were any.
// Out of line: inlined, their registers spill into the FP32 path.  (Whole states
// by all waves, as validity has it, take a second call in the motion's loop:
// 2,000 motions of the 14-joint robot out of range 1,446 -> 1,170 us, but 1,000
// in range 95 -> 103, and 64 against a cloud 41 -> 49.)
__device__ __noinline__ bool edge_decide64(const EdgeKernelArgs* args, const EdgeStates es, int base, int C,
                                           const ValidLds<true> out) {
  const EdgeKernelArgs& A = *args;
  const int lane = threadIdx.x & 63, cfg = lane & (C - 1);
  const bool taylor = A.ka.base_type == PMP_BASE_FIXED;
  auto point = [&](int i) { return es.at(A.ea, min(base + i, es.n_wp - 1)); };
  const bool any = decide_pending(lane, cfg, A.ka, A.k64, A.s64, taylor, out, point);
  const bool whole = decide_whole(lane, cfg, lane / C, kBlockSpheres * C / 64, 0, 1, A.k64, A.s64, taylor,
                                  base + cfg < es.n_wp, out, point);
  wave_lds_order();
  return wave_any(any || whole);
}

template <bool kCloud>
__global__ void __launch_bounds__(1024) edges_staged_kernel(EdgeKernelArgs args) {
  HIP_DYNAMIC_SHARED(float, staged_lds)
  const int D = args.ka.n_cols, lane = threadIdx.x & 63;
  const EdgeLds el = args.el;
  ValidLds<true> out;
  out.flags = reinterpret_cast<int*>(staged_lds + el.flags);
  out.count = out.flags + 64;
  int* queue = out.count + 1;
  out.first = queue + 1;
  out.pend = out.first + 1;
  double* ends = reinterpret_cast<double*>(staged_lds + el.flags + 64 + 4 + 3 * kPendMax);
  edge_begin<true>(args.ea);
  // Workgroups go to the XCDs in turn; each XCD takes a contiguous range of a
  // round's motions, whose endpoints share cache lines.
  const int g = (int)blockIdx.x, n = (int)gridDim.x, x = g % kXcds;
  const int at = x * (n / kXcds) + min(x, n % kXcds) + g / kXcds;
  for (int64_t e0 = 0; e0 < args.ea.E; e0 += n) {
    const int left = (int)min((int64_t)n, args.ea.E - e0);
    if (at >= left) break;
    const int64_t e = e0 + at;
    if (e0 > 0) __syncthreads();  // the last motion's results have been read
    double a = 0.0, b = 0.0, width = 0.0, inv_width = 0.0;
    if (lane < D) {
      a = args.ea.s1[(int64_t)lane * args.ea.lds + e];
      b = args.ea.s2[(int64_t)lane * args.ea.lds + e];
      width = args.ea.width[lane];
      inv_width = args.ea.inv_width[lane];
      if (threadIdx.x < 64) {
        ends[lane] = a;
        ends[D + lane] = b;
      }
    }
    const double ratio = edge_step_ratio(args.ea, D, a, b, width, inv_width);
    __syncthreads();
    int state = 1, checked = 0;
    bool redone = false;
    if (wave_any(ratio != INFINITY)) {
      if (wave_any(!(ratio > 0.0) || 1.0 / ratio > kMaxEdgeStates)) {  // NaN states, or more than a motion may hold
        state = 0;
        checked = -1;
      } else {
        const EdgeStates es{ends, D, __builtin_amdgcn_readfirstlane((int)floor(1.0 / ratio) + 1), ratio};
        checked = es.n_wp;
        for (int base = 0; base < es.n_wp;) {
          const int left = es.n_wp - base, h = max(el.h_min, left <= 8 ? 8 : (left <= 16 ? 4 : (left <= 32 ? 2 : 1)));
          const int C = 64 / h;
          if (h == 1)
            edge_chunk<kCloud, 1>(staged_lds, es, base, out, queue);
          else if (h == 2)
            edge_chunk<kCloud, 2>(staged_lds, es, base, out, queue);
          else if (h == 4)
            edge_chunk<kCloud, 4>(staged_lds, es, base, out, queue);
          else
            edge_chunk<kCloud, 8>(staged_lds, es, base, out, queue);
          if (threadIdx.x < 64 && edge_decide64(&args_again<EdgeKernelArgs>(), es, base, C, out))
            redone = true;
          // only the first wave needs the last chunk's answer
          if (C < left) __syncthreads();
          const int first = __builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile int*>(out.first));
          if (first != INT_MAX) {
            state = 0;
            checked = base + first + 1;
            break;
          }
          base += C;
          if (base < es.n_wp) __syncthreads();  // every wave has read `first`
        }
      }
    }
    if (threadIdx.x == 0) {
      args.ea.valid[e] = (uint8_t)state;
      if (args.ea.n_checked) args.ea.n_checked[e] = checked;
      if (redone) atomicAdd(args.ea.counter + kCntStaged + args.ea.slot, 1);
    }
  }
  if (threadIdx.x == 0) edge_clock_end(args.ea);
}

hipError_t launch_edges_staged(const KinArgs<float>& k32, const KinArgs<double>& k64, const SceneArgs<float>& s32,
                               const SceneArgs<double>& s64, const EdgeArgs& ea, float band, int waves, int block,
                               hipStream_t st) {
  EdgeLds el{};
  size_t lds = 0;
  for (el.h_min = 1;; el.h_min *= 2) {
    const StageLds L = stage_lds(k32, 64 / el.h_min);
    const int keep = k64.slot_wave_bytes / (int)sizeof(float);  // one wave's FP64 kept poses
    el.flags = ((L.end < keep ? keep : L.end) + 1) & ~1;
    lds = sizeof(float) * (size_t)(el.flags + 64 + 4 + 3 * kPendMax + 4 * k32.n_cols);
    if (lds <= (size_t)k32.lds_limit) break;
    if (el.h_min == 8) return hipErrorInvalidConfiguration;  // 8 states of any robot fit
  }
  // 8 waves while a motion has a CU to itself, self pairs to share out or a cloud,
  // else 4 (7R arm, 512 motions of a tenth of the joint range: 20 us, 25 with 8
  // waves, 42 with 16; with self pairs, 14 joints, 1,024: 119 with 8, 145 with 4;
  // 4,096: 332 with 4, 346 with 8; clouds, 7R arm, 16,384: 584 with 4, 911 with 8;
  // 14 joints 2,845 and 2,394); 16 where the tables leave a CU one workgroup (31
  // joints, 1,024: 145 with 16, 167 with 8; 60 joints 273 and 328)
  const bool wide = ea.E <= kCus || (s32.n_cloud > 0 && (ea.E <= 32 * kCus || staged_fit(k32) < 4)) ||
                    (k32.n_pairs > 0 && ea.E <= 8 * kCus);
  const int W = block > 0 ? block / 64 : (2 * lds > (size_t)k32.lds_limit ? 16 : (wide ? 8 : 4));
  const int64_t most = waves > 0 ? (waves < W ? 1 : waves / W) : 1 << 20;
  return launch_last(s32.n_cloud > 0 ? edges_staged_kernel<true> : edges_staged_kernel<false>,
                     dim3((unsigned)(ea.E < most ? ea.E : most)), dim3(64 * W), lds, st,
                     EdgeKernelArgs{k32, s32, k64, s64, ea, el, band});
}

}  // namespace pmp
