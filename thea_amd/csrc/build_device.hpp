// Device pieces shared by the single-mesh build (build.hip) and the batched plan (batch.hip): the box
// pyramid over sorted elements and the per-triangle records.
#pragma once

#include "kernels_common.hpp"
#include "query.hpp"
#include "tri_math.hpp"

namespace thg {

constexpr int PYR_BLOCK = 256;

__device__ __forceinline__ void pyramid_put(const BoxLevels &P, int level, int64_t i, float3 lo, float3 hi) {
  if (level > P.top || i >= P.count(level)) return;
  float4 *b = P.box + 2 * (P.off[level] + i);
  b[0] = make_float4(lo.x, lo.y, lo.z, 0.0f);
  b[1] = make_float4(hi.x, hi.y, hi.z, 0.0f);
}

__device__ __forceinline__ float3 min3(float3 a, float3 b) { return f3(fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z)); }
__device__ __forceinline__ float3 max3(float3 a, float3 b) { return f3(fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z)); }
__device__ __forceinline__ float3 shfl_xor3(float3 v, int m) {
  return f3(__shfl_xor(v.x, m, WAVE), __shfl_xor(v.y, m, WAVE), __shfl_xor(v.z, m, WAVE));
}

// Stores the boxes of a 256-thread block's elements (thread t: element 256 blockIdx.x + t) at level
// `base` of the pyramid (if store_base) and of their aligned runs at the next 8 levels.
__device__ __forceinline__ void pyramid_block(const BoxLevels &P, int base, bool store_base, float3 lo, float3 hi) {
  __shared__ float3 s_lo[PYR_BLOCK / WAVE], s_hi[PYR_BLOCK / WAVE];
  const int64_t idx = (int64_t)blockIdx.x * PYR_BLOCK + threadIdx.x;
  if (store_base) pyramid_put(P, base, idx, lo, hi);
#pragma unroll
  for (int L = 1; L <= 6; ++L) {
    lo = min3(lo, shfl_xor3(lo, 1 << (L - 1)));
    hi = max3(hi, shfl_xor3(hi, 1 << (L - 1)));
    if ((threadIdx.x & ((1 << L) - 1)) == 0) pyramid_put(P, base + L, idx >> L, lo, hi);
  }
  if (lane_id() == 0) {
    s_lo[threadIdx.x / WAVE] = lo;
    s_hi[threadIdx.x / WAVE] = hi;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const int w = 2 * threadIdx.x;
    pyramid_put(P, base + 7, 2 * (int64_t)blockIdx.x + threadIdx.x, min3(s_lo[w], s_lo[w + 1]), max3(s_hi[w], s_hi[w + 1]));
  } else if (threadIdx.x == 2) {
    pyramid_put(P, base + 8, blockIdx.x, min3(min3(s_lo[0], s_lo[1]), min3(s_lo[2], s_lo[3])),
                max3(max3(s_hi[0], s_hi[1]), max3(s_hi[2], s_hi[3])));
  }
}

// Ray record of a triangle (RayTri), its last-of-leaf flag clear.
__device__ __forceinline__ RayTri make_raytri(float3 v0, float3 v1, float3 v2, float id) {
  const float3 e01 = sub3(v1, v0), e02 = sub3(v2, v0);
  RayTri o;
  o.a = make_float4(v0.x, v0.y, v0.z, id);
  o.b = make_float4(e01.x, e01.y, e01.z, 0.0f);
  o.c = make_float4(e02.x, e02.y, e02.z, 0.0f);
  return o;
}

// Records of one triangle in leaf order and its box in the pyramid. One kernel writes all of them
// from registers: three kernels, two of them reading the 128-byte records back, took 104 us for
// 1M triangles, this one takes 80 us with the pyramid's lower levels (208 bytes written per triangle).
__device__ __forceinline__ void put_triangle(int64_t k, float3 v0, float3 v1, float3 v2, int32_t id,
                                             TriRec *__restrict__ rec, RayTri *__restrict__ ray,
                                             ScreenRec *__restrict__ scr) {
  const TriRec r = make_trirec(v0, v1, v2, id);
  rec[k] = r;
  if (ray) ray[k] = make_raytri(v0, v1, v2, r.pl.w);
  ScreenRec sc;
  sc.c = r.sb;
  sc.n = make_float4(r.p0.w, r.p1.w, r.p2.w, 0.0f);
  scr[k] = sc;
}

}  // namespace thg
