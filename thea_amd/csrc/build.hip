// LBVH construction on the GPU (replaces Thea's kd-tree build, Algorithms/BvhN.hpp:1366-1525).
//
//  1. k_elem_prep     element boxes and centres (triangle: Thea's centroid formula (v0+v1+v2)/3,
//                     Triangle3.hpp:148; point: the point), per-block bounds reduced by one more
//                     small kernel (ordered-int min/max).
//  2. k_morton        30-bit Morton code of each centre in the centre bounds.
//  3. radix sort      (code, element) pairs, stable, so equal codes keep element order.
//  4. k_karras        binary radix tree over the sorted codes (Karras, "Maximizing Parallelism in
//                     the Construction of BVHs, Octrees, and k-d Trees", HPG 2012), duplicate codes
//                     disambiguated by position; nodes of more than leaf_size elements are kept.
//  5. k_tri_records, k_point_records
//                     element records in leaf order (TriRec with Thea's per-triangle constants,
//                     RayTri, ScreenRec) and the box pyramid: the boxes of every aligned run of 2^L
//                     sorted elements, a block's 256 at a time from registers.
//  6. k_emit          kept nodes compacted into 64-byte BNodes holding both children's boxes. A
//                     node is a range of sorted elements, so its box is the union of the at most
//                     2 log2(range) pyramid runs that tile it.
//  7. k_node_depth    levels of the compacted tree.
// Boxes are exact float min/max of element coordinates; the query kernels add their own rounding
// slack, so no padding is applied here.
#include "kernels_common.hpp"
#include "build_device.hpp"
#include "query.hpp"
#include "tri_math.hpp"

namespace thg {

constexpr int B_BLOCK = 256;

struct BoundsAcc {  // ordered-int encoded: elem lo xyz, elem hi xyz, centre lo xyz, centre hi xyz
  int v[12];
};

__device__ __forceinline__ float3 ld_vert(const float *__restrict__ verts, int64_t i) {
  return f3(verts[3 * i], verts[3 * i + 1], verts[3 * i + 2]);
}

__global__ void __launch_bounds__(B_BLOCK) k_elem_prep(const float *__restrict__ verts, const int32_t *__restrict__ tris,
                                                       int64_t n, int points, float4 *__restrict__ center,
                                                       int *__restrict__ part) {
  float mn[6] = {INFINITY, INFINITY, INFINITY, INFINITY, INFINITY, INFINITY};
  float mx[6] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY};
  for (int64_t i = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x; i < n; i += (int64_t)gridDim.x * B_BLOCK) {
    float3 lo, hi, c;
    if (points) {
      c = ld_vert(verts, i);
      lo = c;
      hi = c;
    } else {
      float3 v0 = ld_vert(verts, tris[3 * i]), v1 = ld_vert(verts, tris[3 * i + 1]), v2 = ld_vert(verts, tris[3 * i + 2]);
      lo = f3(fminf(v0.x, fminf(v1.x, v2.x)), fminf(v0.y, fminf(v1.y, v2.y)), fminf(v0.z, fminf(v1.z, v2.z)));
      hi = f3(fmaxf(v0.x, fmaxf(v1.x, v2.x)), fmaxf(v0.y, fmaxf(v1.y, v2.y)), fmaxf(v0.z, fmaxf(v1.z, v2.z)));
      float3 s = add3(add3(v0, v1), v2);
      c = f3(s.x / 3.0f, s.y / 3.0f, s.z / 3.0f);
    }
    center[i] = make_float4(c.x, c.y, c.z, 0.0f);
    mn[0] = fminf(mn[0], lo.x); mn[1] = fminf(mn[1], lo.y); mn[2] = fminf(mn[2], lo.z);
    mx[0] = fmaxf(mx[0], hi.x); mx[1] = fmaxf(mx[1], hi.y); mx[2] = fmaxf(mx[2], hi.z);
    mn[3] = fminf(mn[3], c.x); mn[4] = fminf(mn[4], c.y); mn[5] = fminf(mn[5], c.z);
    mx[3] = fmaxf(mx[3], c.x); mx[4] = fmaxf(mx[4], c.y); mx[5] = fmaxf(mx[5], c.z);
  }
  // Block partials in BoundsAcc's slot order (no same-address atomics: they serialise in L2).
  __shared__ float red[B_BLOCK / WAVE][12];
  const int w = threadIdx.x / WAVE;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const float a = wave_min(mn[k]), b = wave_max(mx[k]);
    if (lane_id() == 0) {
      red[w][k < 3 ? k : 6 + (k - 3)] = a;
      red[w][k < 3 ? 3 + k : 9 + (k - 3)] = b;
    }
  }
  __syncthreads();
  if (threadIdx.x < 12) {
    const int k = threadIdx.x;
    const bool lo_slot = k < 3 || (k >= 6 && k < 9);
    float v = red[0][k];
    for (int ww = 1; ww < B_BLOCK / WAVE; ++ww) v = lo_slot ? fminf(v, red[ww][k]) : fmaxf(v, red[ww][k]);
    part[(int64_t)blockIdx.x * 12 + k] = float_to_ord(v);
  }
}

// One wave per slot: the min (lo slots) or max (hi slots) of the block partials.
// Also clears the depth, sets the words of a single-leaf tree (one: its node count and even-depth flag,
// zero: the flag's scan and the position of a lone element) and marks node 0 as the root.
__global__ void __launch_bounds__(12 * WAVE) k_bounds_reduce(const int *__restrict__ part, int nb,
                                                             BoundsAcc *__restrict__ acc, int32_t *__restrict__ depth,
                                                             uint32_t *__restrict__ one, uint32_t *__restrict__ zero,
                                                             int32_t *__restrict__ parent) {
  const int k = threadIdx.x / WAVE, lane = lane_id();
  if (threadIdx.x == 0) {
    *depth = 0;
    *one = 1;
    *zero = 0;
    parent[0] = -1;
  }
  const bool lo_slot = k < 3 || (k >= 6 && k < 9);
  int v = lo_slot ? float_to_ord(INFINITY) : float_to_ord(-INFINITY);
  for (int b = lane; b < nb; b += WAVE) {
    const int x = part[(int64_t)b * 12 + k];
    v = lo_slot ? min(v, x) : max(v, x);
  }
  for (int off = 32; off >= 1; off >>= 1) {
    const int o = __shfl_xor(v, off, WAVE);
    v = lo_slot ? min(v, o) : max(v, o);
  }
  if (lane == 0) acc->v[k] = v;
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v &= 0x3FF;
  v = (v | (v << 16)) & 0x030000FF;
  v = (v | (v << 8)) & 0x0300F00F;
  v = (v | (v << 4)) & 0x030C30C3;
  v = (v | (v << 2)) & 0x09249249;
  return v;
}

__device__ __forceinline__ uint32_t morton30(float3 c, float3 lo, float3 inv) {
  float x = (c.x - lo.x) * inv.x, y = (c.y - lo.y) * inv.y, z = (c.z - lo.z) * inv.z;
  uint32_t ix = (uint32_t)fminf(fmaxf(x * 1024.0f, 0.0f), 1023.0f);
  uint32_t iy = (uint32_t)fminf(fmaxf(y * 1024.0f, 0.0f), 1023.0f);
  uint32_t iz = (uint32_t)fminf(fmaxf(z * 1024.0f, 0.0f), 1023.0f);
  return (spread10(ix) << 2) | (spread10(iy) << 1) | spread10(iz);
}

// Morton codes in the centre bounds (acc) and the histograms of their first sorted digit, one sort
// tile per block.
template <int ITEMS>
__global__ void __launch_bounds__(RS_BLOCK) k_morton(const float4 *__restrict__ center, int64_t n,
                                                     const BoundsAcc *__restrict__ acc, uint32_t tiles,
                                                     uint32_t *__restrict__ keys, uint32_t *__restrict__ hist) {
  __shared__ RadixHist h;
  h.clear();
  float f[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) f[k] = ord_to_float(acc->v[6 + k]);
  const float3 lo = f3(f[0], f[1], f[2]), ext = f3(f[3] - f[0], f[4] - f[1], f[5] - f[2]);
  const float3 inv = f3(ext.x > 0 ? 1.0f / ext.x : 0.0f, ext.y > 0 ? 1.0f / ext.y : 0.0f,
                        ext.z > 0 ? 1.0f / ext.z : 0.0f);
  const int64_t base = (int64_t)blockIdx.x * (RS_BLOCK * ITEMS);
#pragma unroll 4
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t i = base + (int64_t)r * RS_BLOCK + threadIdx.x;
    if (i < n) {
      const float4 c = center[i];
      const uint32_t key = morton30(f3(c.x, c.y, c.z), lo, inv);
      keys[i] = key;
      h.count(key, 0);
    }
  }
  h.store(hist, tiles);
}

// Common prefix length of sorted (code, position) keys i and j; -1 outside [0, n).
__device__ __forceinline__ int delta(const uint32_t *__restrict__ k, int64_t n, int64_t i, int64_t j) {
  if (j < 0 || j >= n) return -1;
  uint32_t a = k[i], b = k[j];
  if (a == b) return 32 + __clz((uint32_t)i ^ (uint32_t)j);
  return __clz(a ^ b);
}

// Internal node i of n - 1: its range [first, last], its split g (left child [first, g], right child
// [g + 1, last]; bit 31 set if i is the range's end) and whether it is kept. Its children, where they
// are internal, are the nodes g and g + 1.
__global__ void __launch_bounds__(B_BLOCK) k_karras(const uint32_t *__restrict__ k, int64_t n, int leaf_size,
                                                    int32_t *__restrict__ rfirst, int32_t *__restrict__ rlast,
                                                    uint32_t *__restrict__ split, uint32_t *__restrict__ keep) {
  int64_t i = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  if (i >= n - 1) return;
  int d = (delta(k, n, i, i + 1) - delta(k, n, i, i - 1)) >= 0 ? 1 : -1;
  int dmin = delta(k, n, i, i - d);
  int64_t lmax = 2;
  while (delta(k, n, i, i + lmax * d) > dmin) lmax *= 2;
  int64_t l = 0;
  for (int64_t t = lmax / 2; t >= 1; t /= 2)
    if (delta(k, n, i, i + (l + t) * d) > dmin) l += t;
  int64_t j = i + l * d;
  int dnode = delta(k, n, i, j);
  int64_t s = 0;
  int64_t div = 2;
  int64_t t;
  do {
    t = (l + div - 1) / div;
    if (t >= 1 && delta(k, n, i, i + (s + t) * d) > dnode) s += t;
    div *= 2;
  } while (t > 1);
  int64_t g = i + s * d + (d < 0 ? -1 : 0);
  int64_t first = i < j ? i : j, last = i < j ? j : i;
  rfirst[i] = (int32_t)first;
  rlast[i] = (int32_t)last;
  split[i] = (uint32_t)g | (d < 0 ? 0x80000000u : 0u);
  keep[i] = last - first + 1 > leaf_size ? 1u : 0u;
}

// Levels base + 1 .. base + 8 from level base.
__global__ void __launch_bounds__(B_BLOCK) k_pyramid(BoxLevels P, int base) {
  const int64_t i = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  float3 lo = f3(INFINITY, INFINITY, INFINITY), hi = f3(-INFINITY, -INFINITY, -INFINITY);
  if (i < P.count(base)) {
    const float4 a = P.box[2 * (P.off[base] + i)], b = P.box[2 * (P.off[base] + i) + 1];
    lo = f3(a.x, a.y, a.z);
    hi = f3(b.x, b.y, b.z);
  }
  pyramid_block(P, base, false, lo, hi);
}

BoxLevels box_levels(int64_t n, float4 *box) {
  BoxLevels P{};
  P.n = n;
  P.box = box;
  while (((int64_t)2 << P.top) <= n) ++P.top;
  for (int L = 0; L < P.top; ++L) P.off[L + 1] = P.off[L] + P.count(L);
  return P;
}
int64_t box_level_entries(int64_t n) {
  const BoxLevels P = box_levels(n, nullptr);
  return P.off[P.top] + P.count(P.top);
}

void launch_pyramid_top(const BoxLevels &P, hipStream_t s) {
  for (int base = 8; base < P.top; base += 8) {
    hipLaunchKernelGGL(k_pyramid, dim3(ceil_div(P.count(base), B_BLOCK)), dim3(B_BLOCK), 0, s, P, base);
    launch_check("k_pyramid");
  }
}

// Union of the element boxes of sorted positions [first, last].
__device__ __forceinline__ void range_box(const BoxLevels &P, int64_t first, int64_t last, float3 &lo, float3 &hi) {
  lo = f3(INFINITY, INFINITY, INFINITY);
  hi = f3(-INFINITY, -INFINITY, -INFINITY);
  int64_t l = first, r = last + 1;
  for (int L = 0; l < r; ++L, l >>= 1, r >>= 1) {
    const float4 *b = P.box + 2 * P.off[L];
    if (l & 1) {
      const float4 x = b[2 * l], y = b[2 * l + 1];
      lo = min3(lo, f3(x.x, x.y, x.z));
      hi = max3(hi, f3(y.x, y.y, y.z));
      ++l;
    }
    if (r & 1) {
      --r;
      const float4 x = b[2 * r], y = b[2 * r + 1];
      lo = min3(lo, f3(x.x, x.y, x.z));
      hi = max3(hi, f3(y.x, y.y, y.z));
    }
  }
}

// Emit the collapsed tree. `fidx` = exclusive prefix of keep (final node index of kept nodes, plus
// `base`); a child that is not kept becomes a leaf over its whole element range. parent[node] = the
// parent's final index, for every kept node but the roots.
//
// Each box is read from the pyramid (a handful of 32-byte runs, most ranges being short) instead of
// being merged bottom-up: the walks of a refit, one element per thread to the next unfinished ancestor
// and fenced above 1,024 elements, took 285 us of a 1M-triangle build, where this kernel takes 41 us
// (17 us without boxes) and the pyramid's upper levels 10 us, and needed parent links, arrival counters
// and a box per internal node (96-mesh plan: 502 -> 117 us).
__global__ void __launch_bounds__(B_BLOCK) k_emit(int64_t ni, int32_t base, const uint32_t *__restrict__ keep,
                                                  const uint32_t *__restrict__ fidx, const int32_t *__restrict__ rfirst,
                                                  const int32_t *__restrict__ rlast,
                                                  const uint32_t *__restrict__ split, BoxLevels P,
                                                  BNode *__restrict__ out, int32_t *__restrict__ parent) {
  const int64_t i = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  if (i >= ni || !keep[i]) return;
  const uint32_t sp = split[i];
  const int64_t first = rfirst[i], last = rlast[i], g = sp & 0x7fffffffu;
  const int64_t shift = i - ((sp >> 31) ? last : first);  // node index less sorted position (batched trees)
  float3 lo[2], hi[2];
  int32_t ref[2], cnt[2];
  const int32_t me = base + (int32_t)fidx[i];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int64_t a = c == 0 ? first : g + 1, b = c == 0 ? g : last;
    const int64_t node = g + c + shift;
    range_box(P, a, b, lo[c], hi[c]);
    if (a == b || !keep[node]) {
      ref[c] = ~(int32_t)a;
      cnt[c] = (int32_t)(b - a + 1);
    } else {
      ref[c] = base + (int32_t)fidx[node];
      cnt[c] = 0;
      parent[ref[c]] = me;
    }
  }
  BNode nd;
  nd.a = make_float4(lo[0].x, lo[0].y, lo[0].z, hi[0].x);
  nd.b = make_float4(hi[0].y, hi[0].z, lo[1].x, lo[1].y);
  nd.c = make_float4(lo[1].z, hi[1].x, hi[1].y, hi[1].z);
  nd.d = make_int4(ref[0], ref[1], cnt[0], cnt[1]);
  out[me] = nd;
}

// Levels of the compacted tree (nodes [first, first + *count)): *max_depth becomes the largest number
// of nodes on a path, which is the depth of the deepest leaf; even[i] (optional) = 1 for nodes at even
// depth.
__global__ void __launch_bounds__(B_BLOCK) k_node_depth(int64_t first, const uint32_t *__restrict__ count,
                                                        const int32_t *__restrict__ parent,
                                                        int32_t *__restrict__ max_depth, uint32_t *__restrict__ even) {
  const int64_t k = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  int d = 0;
  if (k < (int64_t)*count) {
    d = 1;
    for (int32_t p = parent[first + k]; p >= 0; p = parent[p]) ++d;
    if (even) even[k] = d & 1;
  }
  const int m = (int)wave_max((float)d);  // every lane of the wave takes part in the reduction
  // one atomic per wave, and none once the maximum is known to be at least this wave's
  if (lane_id() == 0 && m > __hip_atomic_load(max_depth, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(max_depth, m);
}

__global__ void __launch_bounds__(B_BLOCK) k_tri_records(const float *__restrict__ verts, const int32_t *__restrict__ tris,
                                                         const uint32_t *__restrict__ sorted, int64_t n,
                                                         TriRec *__restrict__ rec, RayTri *__restrict__ ray,
                                                         ScreenRec *__restrict__ scr, BoxLevels P) {
  const int64_t k = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  float3 lo = f3(INFINITY, INFINITY, INFINITY), hi = f3(-INFINITY, -INFINITY, -INFINITY);
  if (k < n) {
    const int64_t e = sorted[k];
    const float3 v0 = ld_vert(verts, tris[3 * e]), v1 = ld_vert(verts, tris[3 * e + 1]),
                 v2 = ld_vert(verts, tris[3 * e + 2]);
    lo = min3(v0, min3(v1, v2));
    hi = max3(v0, max3(v1, v2));
    put_triangle(k, v0, v1, v2, (int32_t)e, rec, ray, scr);
  }
  pyramid_block(P, 0, true, lo, hi);
}

__global__ void __launch_bounds__(B_BLOCK) k_point_records(const float *__restrict__ xyz, const uint32_t *__restrict__ sorted,
                                                           int64_t n, PointRec *__restrict__ out, BoxLevels P) {
  const int64_t k = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  float3 lo = f3(INFINITY, INFINITY, INFINITY), hi = f3(-INFINITY, -INFINITY, -INFINITY);
  if (k < n) {
    const uint32_t e = sorted[k];
    lo = hi = ld_vert(xyz, e);
    PointRec r;
    r.p = make_float4(lo.x, lo.y, lo.z, __int_as_float((int)e));
    out[k] = r;
  }
  pyramid_block(P, 0, true, lo, hi);
}

// Flags the last ray record of every non-empty leaf (RayTri::b.w int bits = 1), so ray traversal can
// run a leaf from its first record without its count.
__global__ void __launch_bounds__(B_BLOCK) k_leaf_ends(const BNode *__restrict__ nodes, int64_t num_nodes,
                                                       RayTri *__restrict__ rays) {
  const int64_t i = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  if (i >= num_nodes) return;
  const int4 d = nodes[i].d;
  if (d.x < 0 && d.z > 0) rays[(int64_t)~d.x + d.z - 1].b.w = __int_as_float(1);
  if (d.y < 0 && d.w > 0) rays[(int64_t)~d.y + d.w - 1].b.w = __int_as_float(1);
}

// Leaf bounds of the mesh BVH's leaves (one thread per node; nodes [0, nsmall + *kept), kept may
// be null for 0): the normal is the normalised sum of the leaf's triangle normals and the centre the
// leaf box's centre, both rounded to float; the half-thickness t and the radius r are then the
// largest vertex offsets from them, in double and rounded up, so the leaf's triangles (convex hulls
// of their vertices) lie inside the stored slab and cylinder whatever the normal is.
__global__ void __launch_bounds__(B_BLOCK) k_leaf_bounds(const BNode *__restrict__ nodes, int64_t nsmall,
                                                         const uint32_t *__restrict__ kept, int64_t max_nodes,
                                                         const TriRec *__restrict__ tr, LeafBound *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * B_BLOCK + threadIdx.x;
  const int64_t count = nsmall + (kept ? (int64_t)*kept : 0);
  if (i >= count || i >= max_nodes) return;
  const BNode nd = nodes[i];
  const float lo6[2][3] = {{nd.a.x, nd.a.y, nd.a.z}, {nd.b.z, nd.b.w, nd.c.x}};
  const float hi6[2][3] = {{nd.a.w, nd.b.x, nd.b.y}, {nd.c.y, nd.c.z, nd.c.w}};
  const int32_t ref[2] = {nd.d.x, nd.d.y}, cnt[2] = {nd.d.z, nd.d.w};
  for (int c = 0; c < 2; ++c) {
    if (ref[c] >= 0 || cnt[c] <= 0) continue;
    const int64_t f = ~(int64_t)ref[c];
    double sx = 0, sy = 0, sz = 0;
    for (int64_t e = f; e < f + cnt[c]; ++e) {
      const float4 p0 = tr[e].p0, p1 = tr[e].p1, p2 = tr[e].p2;
      if (isfinite(p0.w) && isfinite(p1.w) && isfinite(p2.w)) { sx += p0.w; sy += p1.w; sz += p2.w; }
    }
    double nn = sqrt(sx * sx + sy * sy + sz * sz);
    if (!(nn > 1e-30)) { sx = 0; sy = 0; sz = 1; nn = 1; }
    const float nx = (float)(sx / nn), ny = (float)(sy / nn), nz = (float)(sz / nn);
    const float cx = (float)(0.5 * ((double)lo6[c][0] + (double)hi6[c][0]));
    const float cy = (float)(0.5 * ((double)lo6[c][1] + (double)hi6[c][1]));
    const float cz = (float)(0.5 * ((double)lo6[c][2] + (double)hi6[c][2]));
    const double len = sqrt((double)nx * nx + (double)ny * ny + (double)nz * nz);
    double t = 0, r2 = 0;
    for (int64_t e = f; e < f + cnt[c]; ++e) {
      const float4 pv[3] = {tr[e].p0, tr[e].p1, tr[e].p2};
      for (int k = 0; k < 3; ++k) {
        const double dx = (double)pv[k].x - cx, dy = (double)pv[k].y - cy, dz = (double)pv[k].z - cz;
        const double s = nx * dx + ny * dy + nz * dz;
        t = fmax(t, fabs(s));
        const double sn = s / len;
        r2 = fmax(r2, dx * dx + dy * dy + dz * dz - sn * sn);
      }
    }
    LeafBound lb;
    lb.a = make_float4(cx, cy, cz, (float)(sqrt(fmax(r2, 0.0)) * (1.0 + 1e-6)));
    lb.b = make_float4(nx, ny, nz, (float)(t * (1.0 + 1e-6)));
    out[f] = lb;
  }
}

void launch_leaf_bounds(const BNode *nodes, int64_t nsmall, const uint32_t *kept, int64_t max_nodes, const TriRec *tr,
                        LeafBound *out, hipStream_t s) {
  if (max_nodes <= 0) return;
  hipLaunchKernelGGL(k_leaf_bounds, dim3(ceil_div(max_nodes, B_BLOCK)), dim3(B_BLOCK), 0, s, nodes, nsmall, kept,
                     max_nodes, tr, out);
  launch_check("k_leaf_bounds");
}

// Single-leaf tree for n <= leaf_size: child 0 holds every element, child 1 is an empty leaf.
__global__ void k_single_leaf(int64_t n, float3 lo, float3 hi, BNode *out) {
  BNode nd;
  nd.a = make_float4(lo.x, lo.y, lo.z, hi.x);
  nd.b = make_float4(hi.y, hi.z, INFINITY, INFINITY);
  nd.c = make_float4(INFINITY, -INFINITY, -INFINITY, -INFINITY);
  nd.d = make_int4(~0, ~0, (int)n, 0);
  out[0] = nd;
}

// Exclusive scan of n uint32 into out (total in out[n]); uses the radix scan kernel's approach.
// (in and out may be the same array)
__global__ void __launch_bounds__(1024) k_excl_scan_u32(const uint32_t *in, uint32_t *out, int64_t n) {
  __shared__ uint32_t part[1024 / WAVE];
  __shared__ uint32_t carry;
  int t = threadIdx.x;
  if (t == 0) carry = 0;
  __syncthreads();
  for (int64_t base = 0; base < n; base += 1024) {
    int64_t i = base + t;
    uint32_t v = i < n ? in[i] : 0;
    uint32_t inc = wave_incl_scan(v);
    int w = t / WAVE, l = t % WAVE;
    if (l == WAVE - 1) part[w] = inc;
    __syncthreads();
    if (w == 0) {
      uint32_t pv = l < 1024 / WAVE ? part[l] : 0;
      uint32_t pinc = wave_incl_scan(pv);
      if (l < 1024 / WAVE) part[l] = pinc - pv;
    }
    __syncthreads();
    uint32_t excl = carry + part[w] + inc - v;
    if (i < n) out[i] = excl;
    __syncthreads();
    if (t == 1023) carry = excl + v;
    __syncthreads();
  }
  if (t == 0) out[n] = carry;
}

// Three-phase exclusive scan of n uint32 (out[n] = total): block sums, scan of the sums, block
// rescan. `sums` must hold ceil(n / 1024) + 1 words.
__global__ void __launch_bounds__(1024) k_scan_block_sums(const uint32_t *__restrict__ in, int64_t n,
                                                          uint32_t *__restrict__ sums) {
  __shared__ uint32_t part[1024 / WAVE];
  int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  uint32_t v = i < n ? in[i] : 0;
  uint32_t s = wave_sum(v);
  if (lane_id() == 0) part[threadIdx.x / WAVE] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < 1024 / WAVE; ++w) t += part[w];
    sums[blockIdx.x] = t;
  }
}

__global__ void __launch_bounds__(1024) k_scan_block_apply(const uint32_t *__restrict__ in, int64_t n,
                                                           const uint32_t *__restrict__ offs, uint32_t *__restrict__ out) {
  __shared__ uint32_t part[1024 / WAVE];
  int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  uint32_t v = i < n ? in[i] : 0;
  uint32_t inc = wave_incl_scan(v);
  int w = threadIdx.x / WAVE;
  if (lane_id() == WAVE - 1) part[w] = inc;
  __syncthreads();
  uint32_t off = offs[blockIdx.x];
  for (int k = 0; k < w; ++k) off += part[k];
  if (i < n) out[i] = off + inc - v;
  if (i == n - 1) out[n] = off + inc;
}

size_t scan_tmp_words(int64_t n) { return (size_t)ceil_div((uint64_t)std::max<int64_t>(n, 1), 1024) + 1; }

void scan_excl_u32(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *tmp, hipStream_t s) {
  if (n <= 0) return;
  uint32_t nb = ceil_div((uint64_t)n, 1024);
  hipLaunchKernelGGL(k_scan_block_sums, dim3(nb), dim3(1024), 0, s, in, n, tmp);
  launch_check("k_scan_block_sums");
  hipLaunchKernelGGL(k_excl_scan_u32, dim3(1), dim3(1024), 0, s, tmp, tmp, (int64_t)nb);
  launch_check("k_excl_scan_u32");
  hipLaunchKernelGGL(k_scan_block_apply, dim3(nb), dim3(1024), 0, s, in, n, tmp, out);
  launch_check("k_scan_block_apply");
}

// Entry points for the batched many-mesh pipeline (batch.hip), which reuses these kernels over
// concatenated meshes with global element positions and node indices.
void launch_emit(int64_t ni, int32_t base, const uint32_t *keep, const uint32_t *fidx, const int32_t *rfirst,
                 const int32_t *rlast, const uint32_t *split, const BoxLevels &P, BNode *out, int32_t *parent,
                 hipStream_t s) {
  if (ni <= 0) return;
  hipLaunchKernelGGL(k_emit, dim3(ceil_div(ni, B_BLOCK)), dim3(B_BLOCK), 0, s, ni, base, keep, fidx, rfirst, rlast,
                     split, P, out, parent);
  launch_check("k_emit");
}

void launch_node_depth(int64_t max_nodes, int64_t first, const uint32_t *count, const int32_t *parent,
                       int32_t *max_depth, uint32_t *even, hipStream_t s) {
  if (max_nodes <= 0) return;
  hipLaunchKernelGGL(k_node_depth, dim3(ceil_div(max_nodes, B_BLOCK)), dim3(B_BLOCK), 0, s, first, count, parent,
                     max_depth, even);
  launch_check("k_node_depth");
}

// Host driver shared by mesh and point builds. Two waits: for the bounds and the kept node count, which
// size the nodes, and for the depth and the ray tree's node count, which sizes that. A tree of one leaf
// knows the latter, and one element needs no sort (one point 163 -> 78 us, four 166 -> 133; with its mesh,
// one triangle 317 -> 176, four 305 -> 217).
void build_bvh(Bvh &b, const float *verts, const int32_t *tris, int64_t n, bool points, int leaf_size, hipStream_t s) {
  b.points = points;
  b.n = n;
  b.leaf_size = leaf_size;
  if (n <= 0) {
    b.num_nodes = 0;
    b.num_leaves = 0;
    b.max_depth = 0;
    return;
  }
  // arrays over the elements that the BVH keeps, in one allocation
  {
    const size_t eb = (size_t)n * (points ? sizeof(PointRec) : sizeof(TriRec));
    Layout lay;
    const size_t oe = lay.add(eb), orr = lay.add(points ? 0 : n * sizeof(RayTri)),
                 os = lay.add(points ? 0 : n * sizeof(ScreenRec)), ol = lay.add(points ? 0 : n * sizeof(LeafBound));
    b.store.alloc(lay.total);
    char *base = b.store.as<char>();
    b.elems.view(base + oe, eb);
    b.rays.view(base + orr, points ? 0 : n * sizeof(RayTri));
    b.screen.view(base + os, points ? 0 : n * sizeof(ScreenRec));
    b.lbounds.view(base + ol, points ? 0 : n * sizeof(LeafBound));
  }
  const int64_t ni = std::max<int64_t>(n - 1, 1);
  const uint32_t grid = std::min<uint32_t>(ceil_div(n, B_BLOCK), 1024);
  struct Counts {  // device words read by the host
    BoundsAcc bounds;
    int32_t depth;
    uint32_t one, zero;
  };
  Layout lay;
  const size_t o_cnt = lay.add(sizeof(Counts)), o_part = lay.add((size_t)grid * 12 * sizeof(int)),
               o_keys = lay.add(n * 4), o_vals = lay.add(n * 4), o_tk = lay.add(n * 4), o_tv = lay.add(n * 4),
               o_hist = lay.add(radix_hist_words(n) * 4), o_first = lay.add(ni * 4), o_last = lay.add(ni * 4),
               o_split = lay.add(ni * 4), o_keep = lay.add(ni * 4), o_fidx = lay.add((ni + 1) * 4),
               o_parent = lay.add(ni * 4), o_stmp = lay.add(scan_tmp_words(ni) * 4),
               // the centres are read before the pyramid is written, the flags of the ray tree written after
               // the pyramid's last use
               o_box = lay.add(std::max<size_t>((size_t)box_level_entries(n) * 32, n * sizeof(float4)));
  Workspace ws;
  ws.alloc(lay.total, s);
  Counts *cnt = ws.at<Counts>(o_cnt);
  float4 *center = ws.at<float4>(o_box);
  uint32_t *keys = ws.at<uint32_t>(o_keys), *vals = ws.at<uint32_t>(o_vals), *hist = ws.at<uint32_t>(o_hist);
  uint32_t *keep = ws.at<uint32_t>(o_keep), *fidx = ws.at<uint32_t>(o_fidx), *stmp = ws.at<uint32_t>(o_stmp);
  int32_t *parent = ws.at<int32_t>(o_parent);

  hipLaunchKernelGGL(k_elem_prep, dim3(grid), dim3(B_BLOCK), 0, s, verts, tris, n, points ? 1 : 0, center,
                     ws.at<int>(o_part));
  launch_check("k_elem_prep");
  hipLaunchKernelGGL(k_bounds_reduce, dim3(1), dim3(12 * WAVE), 0, s, ws.at<int>(o_part), (int)grid, &cnt->bounds,
                     &cnt->depth, &cnt->one, &cnt->zero, parent);
  launch_check("k_bounds_reduce");
  if (n == 1) {
    vals = &cnt->zero;
  } else {
    const uint32_t tiles = radix_tiles(n);
    if (radix_items(n) == RS_ITEMS_SMALL)
      hipLaunchKernelGGL(k_morton<RS_ITEMS_SMALL>, dim3(tiles), dim3(RS_BLOCK), 0, s, center, n, &cnt->bounds, tiles,
                         keys, hist);
    else
      hipLaunchKernelGGL(k_morton<RS_ITEMS_LARGE>, dim3(tiles), dim3(RS_BLOCK), 0, s, center, n, &cnt->bounds, tiles,
                         keys, hist);
    launch_check("k_morton");
    radix_sort_iota(keys, vals, ws.at<uint32_t>(o_tk), ws.at<uint32_t>(o_tv), hist, n, 0, 32, true, s);
  }

  const BoxLevels P = box_levels(n, ws.at<float4>(o_box));
  if (points)
    hipLaunchKernelGGL(k_point_records, dim3(ceil_div(n, B_BLOCK)), dim3(B_BLOCK), 0, s, verts, vals, n,
                       b.elems.as<PointRec>(), P);
  else
    hipLaunchKernelGGL(k_tri_records, dim3(ceil_div(n, B_BLOCK)), dim3(B_BLOCK), 0, s, verts, tris, vals, n,
                       b.elems.as<TriRec>(), b.rays.as<RayTri>(), b.screen.as<ScreenRec>(), P);
  launch_check("k_records");

  const bool single = n <= leaf_size;
  uint32_t kept = 1;
  if (!single) {
    hipLaunchKernelGGL(k_karras, dim3(ceil_div(ni, B_BLOCK)), dim3(B_BLOCK), 0, s, keys, n, leaf_size,
                       ws.at<int32_t>(o_first), ws.at<int32_t>(o_last), ws.at<uint32_t>(o_split), keep);
    launch_check("k_karras");
    scan_excl_u32(keep, fidx, ni, stmp, s);
    launch_pyramid_top(P, s);
    THG_HIP(hipMemcpyAsync(&kept, fidx + ni, 4, hipMemcpyDeviceToHost, s));
  }
  BoundsAcc h;
  THG_HIP(hipMemcpyAsync(&h, &cnt->bounds, sizeof(h), hipMemcpyDeviceToHost, s));
  THG_HIP(hipStreamSynchronize(s));
  float f[12];
  for (int k = 0; k < 12; ++k) f[k] = ord_to_float(h.v[k]);
  b.lo = f3(f[0], f[1], f[2]);
  b.hi = f3(f[3], f[4], f[5]);
  b.scale = 0;
  for (int k = 0; k < 6; ++k) b.scale = std::max(b.scale, std::fabs(f[k]));
  require(std::isfinite(b.scale), "element coordinates must be finite");
  b.nodes.alloc((size_t)kept * sizeof(BNode));
  b.num_nodes = kept;
  b.num_leaves = single ? 1 : (int64_t)kept + 1;  // a full binary tree
  if (single) {
    hipLaunchKernelGGL(k_single_leaf, dim3(1), dim3(1), 0, s, n, b.lo, b.hi, b.nodes.as<BNode>());
    launch_check("k_single_leaf");
  } else {
    launch_emit(ni, 0, keep, fidx, ws.at<int32_t>(o_first), ws.at<int32_t>(o_last), ws.at<uint32_t>(o_split), P,
                b.nodes.as<BNode>(), parent, s);
  }
  // even-depth flags of the nodes and their scan, for the ray tree (in the pyramid's place)
  const uint32_t *even = &cnt->one, *qidx = &cnt->zero;
  uint32_t nq = 1;
  if (!single) {
    uint32_t *flags = points ? nullptr : ws.at<uint32_t>(o_box);
    launch_node_depth(kept, 0, fidx + ni, parent, &cnt->depth, flags, s);
    if (!points) {
      uint32_t *scan = ws.at<uint32_t>(o_first);  // the ranges are no longer needed; o_last follows for the total
      scan_excl_u32(flags, scan, kept, stmp, s);
      THG_HIP(hipMemcpyAsync(&nq, scan + kept, 4, hipMemcpyDeviceToHost, s));
      even = flags;
      qidx = scan;
    }
  }
  if (!points) {
    hipLaunchKernelGGL(k_leaf_ends, dim3(ceil_div(kept, B_BLOCK)), dim3(B_BLOCK), 0, s, b.nodes.as<BNode>(),
                       (int64_t)kept, b.rays.as<RayTri>());
    launch_check("k_leaf_ends");
    launch_leaf_bounds(b.nodes.as<BNode>(), (int64_t)kept, nullptr, (int64_t)kept, b.elems.as<TriRec>(),
                       b.lbounds.as<LeafBound>(), s);
  }
  int32_t depth = 1;
  if (!single) {
    THG_HIP(hipMemcpyAsync(&depth, &cnt->depth, 4, hipMemcpyDeviceToHost, s));
    THG_HIP(hipStreamSynchronize(s));
  }
  b.max_depth = depth;
  if (!points) build_qbvh4(b, even, qidx, nq, s);
  THG_HIP(hipStreamSynchronize(s));
}

}  // namespace thg
