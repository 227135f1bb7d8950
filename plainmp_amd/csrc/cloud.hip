// Sphere-vs-point-cloud distances on the matrix cores.
//
// A cloud is stored as tiles of 64 points (Morton order, so each tile is
// spatially compact) with the tile's AABB and centre o.  For a sphere centre
// c the squared distance to point p is
//     |c - p|^2 = |c - o|^2 + ( |p - o|^2 - 2 (c - o) . (p - o) )
// and the bracket over 16 centres x 16 points is one K = 4 MFMA:
//     A (16 x 4) = [ c - o , 1 ],   B (4 x 16) = [ -2 (p - o) ; |p - o|^2 ].
// Working in tile-local coordinates keeps every term near the tile size; the
// FP32 cancellation error is bounded per tile by kCloudGemmErr (|c'|^2 +
// rho^2) (fk.hpp).  A wave handles 16 queries; a tile is skipped when no
// query's cap reaches the tile's AABB.  (Validity, whose queries are few and
// stop at the first point inside, does not come here: valid.hip.)
#include <float.h>

#include "fk.hpp"
#include "launch.h"

namespace pmp {

typedef float floatx4 __attribute__((ext_vector_type(4)));

// Squared distance between two boxes (0 when they overlap).
__device__ __forceinline__ float box_box_d2(float alx, float aly, float alz, float aux, float auy, float auz,
                                            float blx, float bly, float blz, float bux, float buy, float buz) {
  const float dx = fmaxf(fmaxf(alx - bux, blx - aux), 0.f);
  const float dy = fmaxf(fmaxf(aly - buy, bly - auy), 0.f);
  const float dz = fmaxf(fmaxf(alz - buz, blz - auz), 0.f);
  return dx * dx + dy * dy + dz * dz;
}

__device__ __forceinline__ float wave_min16(float v) {
  for (int s = 1; s < 16; s <<= 1) v = fminf(v, __shfl_xor(v, s, 64));
  return v;
}
__device__ __forceinline__ float wave_max16(float v) {
  for (int s = 1; s < 16; s <<= 1) v = fmaxf(v, __shfl_xor(v, s, 64));
  return v;
}

// min |c - p|^2 over the cloud's tiles for the queries q = e * B + b
// (e < Q / B spheres, b < B configurations); centres in cen[(e * 3 + k) * B +
// b].  Writes out_d2[q] = min squared distance.
//
// A wave takes 16 consecutive spheres of one configuration (spheres are
// ordered by link, so they are close together; consecutive waves take the
// next configurations) and culls by the box around
// its queries grown by their largest reach: 64 super-tiles at a time are
// tested against that box, a lane each, and a ballot lists the survivors;
// then a survivor's tiles, a lane each; a surviving tile is then tested per
// query and, if any query reaches it, compared on the matrix cores.
__global__ void __launch_bounds__(256) cloud_min_kernel(const CloudTile* tiles, const float* tileB,
                                                        const CloudSuper* supers, int super_begin, int n_super,
                                                        const float* cen, const float* cap2, int64_t B, int64_t Q,
                                                        float* out_d2) {
  const int lane = threadIdx.x & 63;
  const int64_t S = Q / B;  // spheres per configuration
  const int64_t groups = (S + 15) / 16;
  // Waves in configuration-fastest order, workgroups handed to the XCDs in
  // turn and each XCD given a contiguous range: neighbouring configurations
  // read the same lines of the [sphere][B] query arrays, in one L2.
  const int g = blockIdx.x, xcd = g % kXcds;
  int64_t first = 0;
  for (int x = 0; x < xcd; ++x) first += ((int64_t)gridDim.x - x + kXcds - 1) / kXcds;
  const int64_t w = (first + g / kXcds) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (w >= groups * B) return;  // wave-uniform
  const int64_t b = w % B, e0 = (w / B) * 16;
  const int i = lane & 15, k = lane >> 4;
  // the A-row query of this lane
  float capi = -1.f;
  if (e0 + i < S) capi = cap2 ? cap2[(e0 + i) * B + b] : FLT_MAX;
  if (!__any(capi >= 0.f)) return;
  float cx = 0.f, cy = 0.f, cz = 0.f;
  if (e0 + i < S) {
    const int64_t e = e0 + i;
    cx = cen[(e * 3 + 0) * B + b];
    cy = cen[(e * 3 + 1) * B + b];
    cz = cen[(e * 3 + 2) * B + b];
  }
  // centres of the four output rows 4k + r held by this lane
  float rx[4], ry[4], rz[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t e = e0 + 4 * k + r;
    rx[r] = ry[r] = rz[r] = 0.f;
    if (e < S) {
      rx[r] = cen[(e * 3 + 0) * B + b];
      ry[r] = cen[(e * 3 + 1) * B + b];
      rz[r] = cen[(e * 3 + 2) * B + b];
    }
  }
  float best[4] = {FLT_MAX, FLT_MAX, FLT_MAX, FLT_MAX};
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  {
    // the box around the live queries and their largest cap
    const bool live = capi >= 0.f;
    const float qlx = wave_min16(live ? cx : FLT_MAX), qly = wave_min16(live ? cy : FLT_MAX),
                qlz = wave_min16(live ? cz : FLT_MAX);
    const float qux = wave_max16(live ? cx : -FLT_MAX), quy = wave_max16(live ? cy : -FLT_MAX),
                quz = wave_max16(live ? cz : -FLT_MAX);
    const float cap = wave_max16(capi);
    for (int s0 = 0; s0 < n_super; s0 += 64) {
      bool near = false;
      if (s0 + lane < n_super) {
        const CloudSuper Sv = supers[super_begin + s0 + lane];
        near = box_box_d2(Sv.lb[0], Sv.lb[1], Sv.lb[2], Sv.ub[0], Sv.ub[1], Sv.ub[2], qlx, qly, qlz, qux, quy, quz) <=
               cap;
      }
      uint64_t smask = __ballot(near);
      while (smask) {
        const int sj = __builtin_ctzll(smask);
        smask &= smask - 1;
        const CloudSuper Su = cload(supers, super_begin + s0 + sj);
        // the super-tile's tiles, a lane each
        bool tnear = false;
        if (lane < Su.count) {
          const CloudTile Tv = tiles[Su.first + lane];
          tnear = box_box_d2(Tv.lb[0], Tv.lb[1], Tv.lb[2], Tv.ub[0], Tv.ub[1], Tv.ub[2], qlx, qly, qlz, qux, quy,
                             quz) <= cap;
        }
        uint64_t tmask = __ballot(tnear);
        while (tmask) {
          const int tj = __builtin_ctzll(tmask);
          tmask &= tmask - 1;
          const int t = Su.first + tj;
          const CloudTile T = cload(tiles, t);
          const float dx = fmaxf(fmaxf(T.lb[0] - cx, cx - T.ub[0]), 0.f);
          const float dy = fmaxf(fmaxf(T.lb[1] - cy, cy - T.ub[1]), 0.f);
          const float dz = fmaxf(fmaxf(T.lb[2] - cz, cz - T.ub[2]), 0.f);
          if (!__any(dx * dx + dy * dy + dz * dz <= capi)) continue;
          const float a = k == 0 ? cx - T.o[0] : (k == 1 ? cy - T.o[1] : (k == 2 ? cz - T.o[2] : 1.f));
          const float* Bt = tileB + (int64_t)t * 256;
          floatx4 d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Bt[lane], zero, 0, 0, 0);
          floatx4 d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Bt[64 + lane], zero, 0, 0, 0);
          floatx4 d2 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Bt[128 + lane], zero, 0, 0, 0);
          floatx4 d3 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Bt[192 + lane], zero, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float ox = rx[r] - T.o[0], oy = ry[r] - T.o[1], oz = rz[r] - T.o[2];
            const float off = ox * ox + oy * oy + oz * oz;
            const float m = fminf(fminf(d0[r], d1[r]), fminf(d2[r], d3[r])) + off;
            best[r] = fminf(best[r], m);
          }
        }
      }
    }
  }
  // minimum over the 16 lanes that share the rows (columns j = lane & 15)
#pragma unroll
  for (int r = 0; r < 4; ++r)
    for (int s = 1; s < 16; s <<= 1) best[r] = fminf(best[r], __shfl_xor(best[r], s, 64));
  if (i == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t e = e0 + 4 * k + r;
      if (e < S) out_d2[e * B + b] = best[r];
    }
  }
}

// clearance[s * B + b] = min(clearance, sqrt(d2) - rc - r_s)
__global__ void __launch_bounds__(256) cloud_clearance_kernel(float* clearance, const float* d2,
                                                              const float* radius_out, float rc, int64_t B,
                                                              int64_t S) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= S * B) return;
  const float v = sqrtf(d2[q]) - rc - radius_out[q / B];
  clearance[q] = fminf(clearance[q], v);
}

hipError_t launch_cloud_clearance(float* clearance, const float* d2, const float* radius_out, float rc, int64_t B,
                                  int64_t S, hipStream_t st) {
  hipLaunchKernelGGL(cloud_clearance_kernel, dim3((unsigned)((S * B + 255) / 256)), dim3(256), 0, st, clearance, d2,
                     radius_out, rc, B, S);
  return hipGetLastError();
}

hipError_t launch_cloud_min(const CloudTile* tiles, const float* tileB, const CloudSuper* supers,
                            const CloudRange& cr, const float* cen, const float* cap2, int64_t B, int64_t Q,
                            float* out_d2, hipStream_t st) {
  const int64_t waves = (Q / B + 15) / 16 * B;  // 16 spheres of one configuration per wave
  hipLaunchKernelGGL(cloud_min_kernel, dim3((unsigned)((waves * 64 + 255) / 256)), dim3(256), 0, st, tiles, tileB,
                     supers, cr.super_begin, cr.n_super, cen, cap2, B, Q, out_d2);
  return hipGetLastError();
}

}  // namespace pmp
