// Host-side interface of the query kernels (query.hip) and sampler (sample.hip).
#pragma once

#include "common.hpp"

namespace thg {

// Batches smaller than this are processed in input order (sorting would cost more than it saves).
constexpr int64_t ORDER_MIN_QUERIES = 4096;

// The work-queue kernels take batches of up to this many queries as they come: their lanes need no
// neighbours, the trees stay in the caches, and hard queries, which an order brings together, fall on
// different waves (100,000 queries on the 20,480-triangle sphere 376 -> 181 us, on the torus of
// 1,048,576 triangles 659 -> 612 us; 200,000 there 919 -> 1,142 us).
constexpr int64_t QUEUE_UNSORTED_MAX = (int64_t)1 << 17;

// Child visiting orders of the compacted closest-point kernel (Bvh::child_order, SegDesc::child_order):
// results never depend on the order, only the work does.
constexpr int CHILD_MAJORITY = 0;  // the child most of the wave's lanes find nearer
constexpr int CHILD_LEADER = 1;    // the child the wave's first active query finds nearer
constexpr int CHILD_BUILD = 2;     // child 0 first

// One batch of a multi-batch launch (k_closest_multi / k_knn_multi / k_ray_multi): the BVH it
// queries, its inputs and outputs, and the first wave of the launch that works on it.
struct SegDesc {
  const void *nodes;
  const void *elems;
  const void *rays;      // RayTri records (ray segments)
  const void *qnodes;    // QNode4 tree (ray segments)
  const float *q;        // queries (closest, k-NN) or ray origins
  const float *q2;       // ray directions
  const uint32_t *order; // optional spatial order of the batch
  const void *screen;    // ScreenRec records (mesh closest-point segments)
  const void *lbounds;   // LeafBound records (mesh closest-point segments; optional)
  int32_t *idx;
  float *cp;             // closest points (closest) / normals (rays)
  float *dist;           // distances (closest, k-NN) / hit times (rays)
  float *d2;
  int64_t n;
  uint64_t wave_begin;
  float best_init;       // squared distance bound (closest, k-NN) / bound on t (rays)
  float scale;
  float max_time;
  int32_t exclude_self;
  int32_t k;
  int32_t points;
  int32_t root;          // node the traversal starts from
  int32_t nelem;         // elements of the segment's tree (k-NN seed window)
  int32_t lanes_log2;    // lanes per query (log2) of the work-queue kernels
  int32_t child_order;   // visiting order of the compacted closest-point kernel (0: majority)
};

// Per-call temporaries of a query batch (spatial order of the queries). By default the sort memory
// is allocated stream-ordered per call; with `ext` set it comes from caller-provided device memory
// (ext_cap queries' worth: 4 * ext_cap words of keys, values and their ping-pong copies, then
// radix_hist_words(ext_cap) histogram words) and nothing is allocated.
struct QueryScratch {
  AsyncBuf keys, vals, tk, tv, hist;
  const uint32_t *order = nullptr;
  uint32_t *ext = nullptr;
  int64_t ext_cap = 0;
  bool timed = true;  // record kernel timing events when the context has timing enabled
  struct Sort {
    uint32_t *keys, *vals, *tk, *tv, *hist;
  };
  Sort sort_memory(int64_t n, hipStream_t s);
  Ctx *timer_ctx(Ctx *c) const { return timed ? c : nullptr; }
};
// Device words a QueryScratch::ext region needs for batches of up to `cap` queries.
size_t sort_scratch_words(int64_t cap);

// Fails with THG_E_INVALID unless every vertex index of the nt triangles (device memory) is in
// [0, nv); synchronises `s`.
void check_tri_indices(const int32_t *tris, int64_t nt, int64_t nv, hipStream_t s);
void build_bvh(Bvh &b, const float *verts, const int32_t *tris, int64_t n, bool points, int leaf_size, hipStream_t s);
// The 4-wide quantized ray tree (Bvh::qnodes) of a built mesh BVH: even[i] = 1 for the nodes at even
// depth, which become its nq nodes, qidx its exclusive scan.
void build_qbvh4(Bvh &b, const uint32_t *even, const uint32_t *qidx, int64_t nq, hipStream_t s);
int order_bits_lo(int64_t n);
void order_queries(const Bvh &b, const float *q, int64_t n, QueryScratch &ws, hipStream_t s);
void order_rays(const Bvh &b, const float *o, const float *d, int64_t n, QueryScratch &ws, hipStream_t s);
float bound_to_best(double dist_bound);
void launch_closest(const Bvh &b, const float *q, int64_t n, double dist_bound, int exclude_self, int32_t *idx,
                    float *cp, float *dist, float *d2, QueryScratch &ws, hipStream_t s);
// Build-pipeline pieces reused by the batched many-mesh plan (batch.hip).
// Leaf bounds of a mesh BVH's leaves into out[first record of each leaf]: nodes [0, nsmall + *kept)
// (kept null: none beyond nsmall), at most max_nodes.
void launch_leaf_bounds(const BNode *nodes, int64_t nsmall, const uint32_t *kept, int64_t max_nodes, const TriRec *tr,
                        LeafBound *out, hipStream_t s);
// The boxes of every aligned run of 2^L sorted elements, L = 0 .. top: run i of level L at
// box[2 (off[L] + i)] (low corner) and the next (high corner). Runs cut short by n are stored but are
// never part of a range.
struct BoxLevels {
  float4 *box;
  int64_t n;
  int64_t off[33];
  int top;
  __host__ __device__ int64_t count(int L) const { return (n + ((int64_t)1 << L) - 1) >> L; }
};
BoxLevels box_levels(int64_t n, float4 *box);
int64_t box_level_entries(int64_t n);
// Levels 9 and up, from level 8 (the record kernels store levels 0 to 8).
void launch_pyramid_top(const BoxLevels &P, hipStream_t s);
// Compacted nodes of the kept internal nodes (k_emit); parent[] of every non-root compacted node.
void launch_emit(int64_t ni, int32_t base, const uint32_t *keep, const uint32_t *fidx, const int32_t *rfirst,
                 const int32_t *rlast, const uint32_t *split, const BoxLevels &P, BNode *out, int32_t *parent,
                 hipStream_t s);
// *max_depth = max(*max_depth, levels) over nodes [first, first + *count); even: see k_node_depth.
void launch_node_depth(int64_t max_nodes, int64_t first, const uint32_t *count, const int32_t *parent,
                       int32_t *max_depth, uint32_t *even, hipStream_t s);
// Exclusive scan of n words: out must hold n + 1 words (the total lands in out[n]) and tmp
// scan_tmp_words(n) words.
size_t scan_tmp_words(int64_t n);
void scan_excl_u32(const uint32_t *in, uint32_t *out, int64_t n, uint32_t *tmp, hipStream_t s);

// Launch many closest-point batches (segments) as one kernel; `seg_dev` is a device copy of the
// descriptor table with wave_begin filled in. Requires every segment's BVH to fit the wave stack.
// concurrent: the launch shares the device with other streams' launches (request server), which
// selects the variant that needs no scratch memory.
// block_waves: waves per workgroup (1, 2, 4, 8); spill_build: the 8-resident-wave build.
void launch_closest_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, bool points, hipStream_t s,
                          bool concurrent = false, int block_waves = 4, bool spill_build = true);
// k <= 16 (longer lists take the work queue).
void launch_knn_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, int k, bool points, hipStream_t s);
// One query per lane over a segment table (stack >= the deepest tree of the segments, at most 64).
void launch_closest_lane_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, bool points, int stack,
                               hipStream_t s);
void launch_knn_lane_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, int k, bool points, int stack,
                           hipStream_t s);
// Closest triangles by work queue: each segment spans ceil(n 2^lanes_log2 / 64) waves.
void launch_closest_queue_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, hipStream_t s);
bool use_queue(int64_t n, int64_t triangles, int max_depth);
bool use_queue_traversal(const Bvh &b, int64_t n);
int queue_lanes_log2(int64_t n);
// k nearest by work queue on mesh BVHs, segments as above.
void launch_knn_queue_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, hipStream_t s);
bool use_knn_queue(const Bvh &b, int64_t n, int k);
int knn_queue_lanes_log2(int64_t n, int k, bool points);
bool use_wave_traversal(const Bvh &b);
// Rays by work queue, segments as above.
void launch_ray_queue_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, hipStream_t s);
bool use_ray_queue(const Bvh &b);
int ray_lanes_log2(int64_t n);
bool order_ray_batch(const Bvh &b, int64_t n);
// One ray per lane on the binary trees; stack: the deepest among the segments plus one (32 or 64
// entries).
void launch_ray_multi(const SegDesc *seg_dev, int nseg, uint64_t total_waves, int stack, hipStream_t s);
// Stack entries a QNode4 walk of one ray in b may need (three per level), and the most that the work
// queue keeps in reserve for it.
inline int q4_stack(const Bvh &b) { return 3 * b.q_depth + 1; }
constexpr int Q4_MAX_STACK = 112;
constexpr int SEG_WAVE_QUERIES = 64;  // queries per wave in the multi-batch kernels
void ray_stats(const Bvh &b, const float *o, const float *d, int64_t n, int32_t *idx, int32_t *counts, hipStream_t s);
void closest_wave_stats(const Bvh &b, const float *q, int64_t n, unsigned long long *stats, QueryScratch &ws,
                        hipStream_t s);
void launch_knn(const Bvh &b, const float *q, int64_t n, int k, double dist_bound, int exclude_self, int32_t *idx,
                float *dist, float *d2, QueryScratch &ws, hipStream_t s);
// Per-wave statistics of the 16-nearest wave kernel on a point BVH (4 int64 per 64-query wave).
void knn_wave_stats(const Bvh &b, const float *q, int64_t n, int exclude_self, int64_t *wstats, QueryScratch &ws,
                    hipStream_t s);
// sort_rays = false traces the rays in input order, for callers whose rays are coherent as they come.
// Results are always written at the rays' input indices.
void launch_ray(const Bvh &b, const float *o, const float *d, int64_t n, float max_time, bool any, int32_t *idx,
                float *t, float *nrm, uint8_t *hit, QueryScratch &ws, hipStream_t s, bool sort_rays = true);

// Sampler
void mesh_cdf(Mesh &m, hipStream_t s);
int64_t launch_sample_approx(Mesh &m, int64_t n, uint64_t seed, uint64_t stream_id, int64_t capacity, float *pos,
                             float *nrm, int32_t *tri, hipStream_t s);
float graph_build(Bvh *b, const float *d_nrm, int md, int64_t trials, uint64_t seed, hipStream_t s, int32_t *d_idx,
                  float *d_sep, int32_t *d_deg, const Bvh *surface = nullptr);
void launch_sample(Mesh &m, int64_t n, uint64_t seed, uint64_t stream_id, float *pos, float *nrm, int32_t *tri,
                   hipStream_t s);

}  // namespace thg
