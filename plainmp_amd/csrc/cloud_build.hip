// Device build of a point cloud's tile tables, the structure the cloud
// distance kernels walk in place of the reference's KD-tree
// (collision/kdtree.cpp:40-65, built by CloudSDF's constructor,
// collision/primitive_sdf.hpp:568-583).
//
// Steps, all on the stream given:
//   1. bounds of the points (two-level min / max, exact in FP64);
//   2. a 30-bit Morton code per point from its position in the bounds
//      (10 bits per axis), packed with the point index as a 64-bit key
//      (code << 30 | index), so that sorting the keys orders the points by
//      code and, within a code, by index;
//   3. three stable counting passes over the code, ten bits each from the low
//      end (the index order is the input's, so it needs no passes): a
//      workgroup takes kSortKeys keys; where its keys of one digit go follows
//      from every workgroup's digit counts and the order within its own;
//   4. one wave per tile of kCloudTile consecutive sorted points: FP64 bounds,
//      the FP32 centre and outward-rounded FP32 bounds, the matrix-core B
//      operands (-2 p', |p'|^2) of the points in tile-local coordinates
//      p' = p - o, and the FP64 world points (padding points far away);
//   5. super-tiles of kCloudSuper consecutive tiles under one FP32 AABB, by the
//      workgroup that writes their tiles.
// Eight dependent launches, each bound by its latency (a scatter pass 14 us, a
// count 4, the tiles 12): 307,200 points 192 -> 73 us, 1,000,000 326 -> 139 (41
// launches before: a bitonic sort over a power of two of keys).  Clouds of at
// most kSortKeys points take two: 1,000 points 31 -> 22 us.
// Every value is a min / max, a rounding of one FP64 operation or a fixed
// sequence of them (no contraction into FMA), so the tables do not depend
// on the launch shape.
#include <float.h>
#include <stdint.h>

#include "launch.h"

#pragma clang fp contract(off)

namespace pmp {

namespace {

constexpr int kBoundsGrid = 256;  // partial bounds: one record of 6 per workgroup
constexpr int64_t kIndexBits = 30;
constexpr int kSortBlock = 512, kSortWaves = kSortBlock / 64;
constexpr int kSortRows = 4;  // keys a thread (100,003 points 49 us, 63 with 8; 600,000 104 and 94)
constexpr int kSortKeys = kSortRows * kSortBlock;
constexpr int kDigitBits = 10, kDigits = 1 << kDigitBits;
constexpr int kSortPasses = 3;
// Up to this many workgroups each scatter pass adds up the counts of all
// workgroups itself (150 for 307,200 points); beyond, a launch of its own does
// so once, the work being quadratic otherwise (307,200 points: the same time
// either way).
constexpr int kSumBlocks = 256;

// Interleave the low 10 bits of v into every third bit.
__device__ inline uint32_t spread10(uint32_t v) {
  v &= 1023u;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// The neighbouring FP32 value towards -inf / +inf of a finite x.
__device__ inline float next_down(float x) {
  if (x == 0.f) return -FLT_TRUE_MIN;
  const int32_t b = __float_as_int(x);
  return __int_as_float(x > 0.f ? b - 1 : b + 1);
}
__device__ inline float next_up(float x) {
  if (x == 0.f) return FLT_TRUE_MIN;
  const int32_t b = __float_as_int(x);
  return __int_as_float(x > 0.f ? b + 1 : b - 1);
}

// Orders a wave's own LDS accesses.
__device__ inline void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Minima in v[0..2], maxima in v[3..5] over the workgroup, in every thread.
__device__ inline void block_bounds(double (&v)[6], double (*red)[6]) {
  for (int m = 32; m > 0; m >>= 1)
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const double o = __shfl_xor(v[k], m);
      v[k] = k < 3 ? fmin(v[k], o) : fmax(v[k], o);
    }
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < 6; ++k) red[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
  for (int k = 0; k < 6; ++k) v[k] = red[0][k];
  for (int w = 1; w < kSortWaves; ++w)
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = k < 3 ? fmin(v[k], red[w][k]) : fmax(v[k], red[w][k]);
}

__global__ void __launch_bounds__(kSortBlock) bounds_kernel(const double* pts, int64_t n, double* part) {
  __shared__ double red[kSortWaves][6];
  double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double x = pts[3 * i + k];
      v[k] = fmin(v[k], x);
      v[3 + k] = fmax(v[3 + k], x);
    }
  block_bounds(v, red);
  if (threadIdx.x < 6) part[6 * blockIdx.x + threadIdx.x] = v[threadIdx.x];
}

// A workgroup's digit counts, two digits a word (at most kSortKeys each).
__device__ inline void write_counts(const uint32_t* hist, uint32_t* counts) {
  __syncthreads();
  counts[(int64_t)blockIdx.x * (kDigits / 2) + threadIdx.x] = hist[2 * threadIdx.x] | (hist[2 * threadIdx.x + 1] << 16);
}
static_assert(kDigits == 2 * kSortBlock, "a thread holds two digits");

// Point (x, y, z)'s code in the bounds v.
__device__ inline uint32_t point_code(const double (&x)[3], const double (&v)[6]) {
  uint32_t c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double lo = v[k], span = v[3 + k] - lo;
    const double u = span > 0 ? (x[k] - lo) / span : 0.0;
    c[k] = (uint32_t)fmin(1023.0, fmax(0.0, u * 1023.0));
  }
  return spread10(c[0]) | (spread10(c[1]) << 1) | (spread10(c[2]) << 2);
}

// The bounds from the partial records, the keys, and the first digit's counts.
__global__ void __launch_bounds__(kSortBlock) keys_kernel(const double* pts, int64_t n, const double* part, int n_part,
                                                          uint64_t* keys, uint32_t* counts) {
  __shared__ double red[kSortWaves][6];
  __shared__ uint32_t hist[kDigits];
  double x[kSortRows][3];
  const int64_t first = (int64_t)blockIdx.x * kSortKeys + threadIdx.x;
#pragma unroll
  for (int r = 0; r < kSortRows; ++r)
#pragma unroll
    for (int k = 0; k < 3; ++k) x[r][k] = first + r * kSortBlock < n ? pts[3 * (first + r * kSortBlock) + k] : 0.0;
  double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
  for (int b = threadIdx.x; b < n_part; b += kSortBlock)
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = k < 3 ? fmin(v[k], part[6 * b + k]) : fmax(v[k], part[6 * b + k]);
  hist[threadIdx.x] = hist[threadIdx.x + kSortBlock] = 0;
  block_bounds(v, red);
#pragma unroll
  for (int r = 0; r < kSortRows; ++r) {
    const int64_t i = first + r * kSortBlock;
    if (i >= n) break;
    const uint32_t code = point_code(x[r], v);
    keys[i] = ((uint64_t)code << kIndexBits) | (uint64_t)i;
    atomicAdd(&hist[code & (kDigits - 1)], 1u);
  }
  write_counts(hist, counts);
}

__device__ inline uint32_t digit_of(uint64_t key, int pass) {
  return (uint32_t)(key >> (kIndexBits + pass * kDigitBits)) & (kDigits - 1);
}

// The counts of a later pass's digit.
__global__ void __launch_bounds__(kSortBlock) counts_kernel(const uint64_t* keys, int64_t n, int pass, uint32_t* counts) {
  __shared__ uint32_t hist[kDigits];
  hist[threadIdx.x] = hist[threadIdx.x + kSortBlock] = 0;
  __syncthreads();
  for (int r = 0; r < kSortRows; ++r) {
    const int64_t i = (int64_t)blockIdx.x * kSortKeys + r * kSortBlock + threadIdx.x;
    if (i < n) atomicAdd(&hist[digit_of(keys[i], pass)], 1u);
  }
  write_counts(hist, counts);
}

// For many workgroups: before[b][d], the keys of digit d in workgroups before
// b, and total[d].  A lane has a word of two digits, a wave a range of b.
__global__ void __launch_bounds__(1024) sums_kernel(const uint32_t* counts, int64_t nb, uint32_t* before,
                                                    uint32_t* total) {
  __shared__ uint2 part[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, word = blockIdx.x * 64 + lane;
  const int64_t lo = nb * w / 16, hi = nb * (w + 1) / 16;
  uint2 s{0, 0};
  for (int64_t b = lo; b < hi; ++b) {
    const uint32_t c = counts[b * (kDigits / 2) + word];
    s.x += c & 0xffffu;
    s.y += c >> 16;
  }
  part[w][lane] = s;
  __syncthreads();
  uint2 at{0, 0};
  for (int u = 0; u < w; ++u) {
    at.x += part[u][lane].x;
    at.y += part[u][lane].y;
  }
  for (int64_t b = lo; b < hi; ++b) {
    const uint32_t c = counts[b * (kDigits / 2) + word];
    before[b * kDigits + 2 * word] = at.x;
    before[b * kDigits + 2 * word + 1] = at.y;
    at.x += c & 0xffffu;
    at.y += c >> 16;
  }
  if (w == 15) {
    total[2 * word] = at.x;
    total[2 * word + 1] = at.y;
  }
}

// The order of a wave's keys among those of the same digit in it: it takes 64
// consecutive keys at a time, the lanes with the same digit find one another by
// ballots, and hist (this wave's, zero) counts the digit's keys so far.
__device__ inline void wave_ranks(const uint64_t (&key)[kSortRows], int live_rows, int pass, uint16_t* hist,
                                  uint32_t (&rank)[kSortRows]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < kSortRows; ++r) {
    const bool live = r < live_rows;
    const uint32_t d = digit_of(key[r], pass);
    uint64_t peers = __ballot(live);
#pragma unroll
    for (int k = 0; k < kDigitBits; ++k) {
      const uint64_t m = __ballot((d >> k) & 1);
      peers &= (d >> k) & 1 ? m : ~m;
    }
    const int pos = __popcll(peers & ((1ull << lane) - 1));
    rank[r] = live ? hist[d] + pos : 0;
    wave_order();
    if (live && pos == 0) hist[d] = (uint16_t)(rank[r] + __popcll(peers));
    wave_order();
  }
}
// Rows of this lane's keys (at first + 64 r) that lie below n.
__device__ inline int live_rows_of(int64_t first, int64_t n) {
  return first < n ? (int)((n - first + 63) / 64 < kSortRows ? (n - first + 63) / 64 : kSortRows) : 0;
}

// Turns the waves' counts into the keys before each wave's (thread t: digits
// 2 t, 2 t + 1), and returns the workgroup's counts.
__device__ inline uint2 wave_prefix(uint16_t (*hist)[kDigits]) {
  uint2 h{0, 0};
  for (int u = 0; u < kSortWaves; ++u) {
    uint16_t* p = hist[u] + 2 * threadIdx.x;
    const uint32_t c0 = p[0], c1 = p[1];
    p[0] = (uint16_t)h.x;
    p[1] = (uint16_t)h.y;
    h.x += c0;
    h.y += c1;
  }
  return h;
}
// Sum of v over the threads before this one.
__device__ inline uint32_t block_before(uint32_t v, uint32_t* wsum) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t incl = v;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const uint32_t o = __shfl_up(incl, s);
    if (lane >= s) incl += o;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  uint32_t at = incl - v;
  for (int u = 0; u < w; ++u) at += wsum[u];
  return at;
}

// One stable pass: the order in the wave, the counts of the waves before, of
// the workgroups before and of the smaller digits say where a key goes.
// before == nullptr: the workgroups' counts are added up here.
__global__ void __launch_bounds__(kSortBlock) scatter_kernel(const uint64_t* in, int64_t n, int pass,
                                                             const uint32_t* counts, const uint32_t* before,
                                                             const uint32_t* total, uint64_t* out) {
  __shared__ uint16_t hist[kSortWaves][kDigits];
  __shared__ uint32_t base[kDigits], all[kDigits];
  __shared__ uint32_t wsum[kSortWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t = threadIdx.x;
  uint64_t key[kSortRows];
  const int64_t first = (int64_t)blockIdx.x * kSortKeys + w * (kSortRows * 64) + lane;
  const int live = live_rows_of(first, n);
#pragma unroll
  for (int r = 0; r < kSortRows; ++r) key[r] = r < live ? in[first + r * 64] : 0;
  for (int i = lane; i < kDigits / 2; i += 64) reinterpret_cast<uint32_t*>(hist[w])[i] = 0;
  if (before) {
    base[2 * t] = before[(int64_t)blockIdx.x * kDigits + 2 * t];
    base[2 * t + 1] = before[(int64_t)blockIdx.x * kDigits + 2 * t + 1];
    all[2 * t] = total[2 * t];
    all[2 * t + 1] = total[2 * t + 1];
  } else {
    const int nb = (int)gridDim.x, me = (int)blockIdx.x;
    uint32_t b0 = 0, b1 = 0, t0 = 0, t1 = 0;
#pragma unroll 16
    for (int b = 0; b < nb; ++b) {
      const uint32_t c = counts[b * (kDigits / 2) + t];
      t0 += c & 0xffffu;
      t1 += c >> 16;
      b0 += b < me ? c & 0xffffu : 0;
      b1 += b < me ? c >> 16 : 0;
    }
    base[2 * t] = b0;
    base[2 * t + 1] = b1;
    all[2 * t] = t0;
    all[2 * t + 1] = t1;
  }
  wave_order();
  uint32_t rank[kSortRows];
  wave_ranks(key, live, pass, hist[w], rank);
  __syncthreads();
  const uint32_t at = block_before(all[2 * t] + all[2 * t + 1], wsum);
  base[2 * t] += at;
  base[2 * t + 1] += at + all[2 * t];
  wave_prefix(hist);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortRows; ++r) {
    const uint32_t d = digit_of(key[r], pass);
    if (r < live) out[base[d] + hist[w][d] + rank[r]] = key[r];
  }
}

// A cloud of one workgroup's keys: bounds, keys and all passes in one launch.
__global__ void __launch_bounds__(kSortBlock) sort_small_kernel(const double* pts, int64_t n, uint64_t* out) {
  __shared__ double red[kSortWaves][6];
  __shared__ uint16_t hist[kSortWaves][kDigits];
  __shared__ uint32_t base[kDigits];
  __shared__ uint32_t wsum[kSortWaves];
  __shared__ uint64_t sorted[kSortKeys];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t = threadIdx.x;
  const int64_t first = w * (kSortRows * 64) + lane;
  const int live = live_rows_of(first, n);
  double x[kSortRows][3], v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
#pragma unroll
  for (int r = 0; r < kSortRows; ++r)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      x[r][k] = r < live ? pts[3 * (first + r * 64) + k] : 0.0;
      if (r < live) {
        v[k] = fmin(v[k], x[r][k]);
        v[3 + k] = fmax(v[3 + k], x[r][k]);
      }
    }
  block_bounds(v, red);
  uint64_t key[kSortRows];
#pragma unroll
  for (int r = 0; r < kSortRows; ++r) key[r] = ((uint64_t)point_code(x[r], v) << kIndexBits) | (uint64_t)(first + r * 64);
  for (int pass = 0; pass < kSortPasses; ++pass) {
    for (int i = lane; i < kDigits / 2; i += 64) reinterpret_cast<uint32_t*>(hist[w])[i] = 0;
    wave_order();
    uint32_t rank[kSortRows];
    wave_ranks(key, live, pass, hist[w], rank);
    __syncthreads();
    const uint2 h = wave_prefix(hist);
    const uint32_t at = block_before(h.x + h.y, wsum);
    base[2 * t] = at;
    base[2 * t + 1] = at + h.x;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRows; ++r) {
      const uint32_t d = digit_of(key[r], pass);
      if (r < live) sorted[base[d] + hist[w][d] + rank[r]] = key[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRows; ++r)
      if (r < live) key[r] = sorted[first + r * 64];
  }
#pragma unroll
  for (int r = 0; r < kSortRows; ++r)
    if (r < live) out[first + r * 64] = key[r];
}

// Tile t by its wave; box: its FP32 bounds.
__device__ inline void tile(const double* pts, int64_t n, const uint64_t* keys, int64_t t, int jj, CloudTile* t32,
                            CloudTile64* t64, float* tb, double* p64, float* box) {
  const int64_t b = t * kCloudTile;
  const bool live = b + jj < n;
  double pw[3] = {0.0, 0.0, 0.0};
  if (live) {
    const int64_t idx = (int64_t)(keys[b + jj] & (((uint64_t)1 << kIndexBits) - 1));
    for (int k = 0; k < 3; ++k) pw[k] = pts[3 * idx + k];
  }
  double lb[3], ub[3], o[3];
  float of[3];
  for (int k = 0; k < 3; ++k) {
    lb[k] = live ? pw[k] : 1e300;
    ub[k] = live ? pw[k] : -1e300;
  }
  for (int m = 32; m > 0; m >>= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lb[k] = fmin(lb[k], __shfl_xor(lb[k], m));
      ub[k] = fmax(ub[k], __shfl_xor(ub[k], m));
    }
  for (int k = 0; k < 3; ++k) {
    o[k] = 0.5 * (lb[k] + ub[k]);
    of[k] = (float)o[k];
  }
  if (jj == 0) {
    CloudTile T;
    CloudTile64 T64;
    for (int k = 0; k < 3; ++k) {
      T64.lb[k] = lb[k];
      T64.ub[k] = ub[k];
      T.o[k] = of[k];
      T.lb[k] = next_down((float)lb[k]);
      T.ub[k] = next_up((float)ub[k]);
      box[k] = T.lb[k];
      box[3 + k] = T.ub[k];
    }
    T.n = (int32_t)((n - b) < kCloudTile ? (n - b) : kCloudTile);
    t32[t] = T;
    t64[t] = T64;
  }
  // B operand [m][k][j] of point 16 m + j, and the FP64 point
  float* col = tb + t * 4 * kCloudTile + (jj / 16) * 64 + (jj % 16);
  double2* pp = reinterpret_cast<double2*>(p64 + (t * kCloudTile + jj) * 4);
  if (live) {
    double pl[3];
    for (int k = 0; k < 3; ++k) pl[k] = (double)(float)(pw[k] - (double)of[k]);
    double n2 = 0.0;
    for (int k = 0; k < 3; ++k) n2 = n2 + pl[k] * pl[k];
    for (int k = 0; k < 3; ++k) col[k * 16] = (float)(-2.0 * pl[k]);
    col[3 * 16] = (float)n2;
    pp[0] = {pw[0], pw[1]};
    pp[1] = {pw[2], 0.0};
  } else {  // padding: never the nearest
    for (int k = 0; k < 3; ++k) col[k * 16] = 0.f;
    col[3 * 16] = 1e30f;
    pp[0] = {1e30, 1e30};
    pp[1] = {1e30, 0.0};
  }
}

// One wave per tile, lane jj with point jj of it, and one workgroup per
// super-tile; tiles and supers are indexed within the cloud, `first` is written
// as tile_base + the cloud's tile index.
__global__ void __launch_bounds__(64 * kCloudSuper) tiles_kernel(const double* pts, int64_t n, const uint64_t* keys,
                                                                 int64_t nt, int32_t tile_base, CloudTile* t32,
                                                                 CloudTile64* t64, float* tb, double* p64,
                                                                 CloudSuper* sup) {
  __shared__ float box[kCloudSuper][6];
  const int64_t t = (int64_t)blockIdx.x * kCloudSuper + (threadIdx.x >> 6);
  const int jj = threadIdx.x & 63;
  if (t < nt) tile(pts, n, keys, t, jj, t32, t64, tb, p64, box[threadIdx.x >> 6]);
  __syncthreads();
  const int64_t a = (int64_t)blockIdx.x * kCloudSuper;
  const int32_t count = (int32_t)((nt - a) < kCloudSuper ? (nt - a) : kCloudSuper);
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    float v = k < 3 ? INFINITY : -INFINITY;
    for (int i = 0; i < count; ++i) v = k < 3 ? fminf(v, box[i][k]) : fmaxf(v, box[i][k]);
    (k < 3 ? sup[blockIdx.x].lb[k] : sup[blockIdx.x].ub[k - 3]) = v;
  } else if (threadIdx.x == 6) {
    sup[blockIdx.x].first = tile_base + (int32_t)a;
    sup[blockIdx.x].count = count;
  }
}
}  // namespace

CloudBuildSizes cloud_build_sizes(int64_t n) {
  CloudBuildSizes z;
  z.n_tiles = (n + kCloudTile - 1) / kCloudTile;
  z.n_supers = (z.n_tiles + kCloudSuper - 1) / kCloudSuper;
  z.n_keys = n;
  const int64_t nb = (n + kSortKeys - 1) / kSortKeys;
  // two buffers of keys, the partial bounds, the counts, and for many
  // workgroups their sums
  z.scratch_bytes = 2 * n * (int64_t)sizeof(uint64_t) + 6 * kBoundsGrid * (int64_t)sizeof(double) +
                    nb * (kDigits / 2) * (int64_t)sizeof(uint32_t);
  if (nb > kSumBlocks) z.scratch_bytes += (nb + 1) * kDigits * (int64_t)sizeof(uint32_t);
  return z;
}

hipError_t launch_cloud_build(const double* pts, int64_t n, int32_t tile_base, CloudTile* t32, CloudTile64* t64,
                              float* tb, double* p64, CloudSuper* sup, void* scratch, hipStream_t st) {
  const CloudBuildSizes z = cloud_build_sizes(n);
  const int64_t nb = (n + kSortKeys - 1) / kSortKeys;
  uint32_t* counts = (uint32_t*)scratch;
  double* part = (double*)(counts + nb * (kDigits / 2));
  uint64_t* keys = (uint64_t*)(part + 6 * kBoundsGrid);
  uint64_t* other = keys + n;
  uint32_t* before = nb > kSumBlocks ? (uint32_t*)(other + n) : nullptr;
  uint32_t* total = before ? before + nb * kDigits : nullptr;
  const dim3 block(kSortBlock), blocks((unsigned)nb);
  if (nb == 1) {
    hipLaunchKernelGGL(sort_small_kernel, dim3(1), block, 0, st, pts, n, keys);
  } else {
    const int64_t want = (n + kSortBlock - 1) / kSortBlock;
    const int grid = (int)(want < kBoundsGrid ? want : kBoundsGrid);
    hipLaunchKernelGGL(bounds_kernel, dim3(grid), block, 0, st, pts, n, part);
    hipLaunchKernelGGL(keys_kernel, blocks, block, 0, st, pts, n, (const double*)part, grid, keys, counts);
    for (int pass = 0; pass < kSortPasses; ++pass) {
      if (pass > 0) hipLaunchKernelGGL(counts_kernel, blocks, block, 0, st, (const uint64_t*)keys, n, pass, counts);
      if (before)
        hipLaunchKernelGGL(sums_kernel, dim3(kDigits / 128), dim3(1024), 0, st, (const uint32_t*)counts, nb, before,
                           total);
      hipLaunchKernelGGL(scatter_kernel, blocks, block, 0, st, (const uint64_t*)keys, n, pass, (const uint32_t*)counts,
                         (const uint32_t*)before, (const uint32_t*)total, other);
      uint64_t* swap = keys;
      keys = other;
      other = swap;
    }
  }
  hipLaunchKernelGGL(tiles_kernel, dim3((unsigned)z.n_supers), dim3(64 * kCloudSuper), 0, st, pts, n,
                     (const uint64_t*)keys, z.n_tiles, tile_base, t32, t64, tb, p64, sup);
  return hipGetLastError();
}

}  // namespace pmp
