// Stable LSD radix sort of 32-bit key/value pairs, 8-bit digits, LDS-staged.
//
// Pass structure (per 8-bit digit):
//   1. k_radix_hist: each tile counts its digits in LDS and writes a 256-entry histogram in
//      digit-major order (hist[d * tiles + tile]). Key kernels that already hold a tile's keys write
//      the first pass's histogram themselves (RadixHist, kernels_common.hpp).
//   2. k_radix_rowscan: one workgroup per digit turns its row of tile counts into exclusive
//      offsets and a row total; the scatter kernel scans the 256 totals itself.
//   3. k_radix_scatter: each wave ranks its contiguous share of the tile on its own (ballots give the
//      rank among equal digits of 64 keys, a wave-private LDS table the counts before them), the
//      tile is put in digit order in LDS and written out in runs of equal digits.
// Used for the 30-bit Morton codes of BVH elements and for spatially ordering query batches.
//
// What bounds it: memory traffic (20 bytes per pair and pass) for millions of pairs, launches below.
// Writing runs from LDS instead of every pair to its own place, and ranking without a block barrier
// per 256 keys (64 barriers per tile before, 4 now), took a pass's scatter over 10M pairs from
// 157 us to 59 us; ordering 10M queries (keys, 3 passes) went from 605 us to
// 273 us, of 100,000 (2 passes) from 93 us to 29 us.
#include "kernels_common.hpp"

namespace thg {

constexpr int RS_WAVES = RS_BLOCK / WAVE;

// Histogram words for any sort of up to n pairs (a smaller sort may use smaller tiles, and so more
// of them than n / its own tile: the small-tile maximum is kept as the floor).
size_t radix_hist_words(int64_t n) {
  const uint64_t m = (uint64_t)std::max<int64_t>(n, 1);
  const uint64_t small = ceil_div(std::min<uint64_t>(m, RS_SMALL_MAX), RS_TILE_SMALL);
  const uint64_t large = m > RS_SMALL_MAX ? ceil_div(m, RS_TILE_LARGE) : 0;
  return (size_t)256 * std::max(small, large) + 256;
}

template <int ITEMS>
__global__ void __launch_bounds__(RS_BLOCK) k_radix_hist(const uint32_t *__restrict__ keys, int64_t n, int shift,
                                                         uint32_t tiles, uint32_t *__restrict__ hist) {
  __shared__ RadixHist h;
  h.clear();
  const int64_t base = (int64_t)blockIdx.x * (RS_BLOCK * ITEMS);
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int64_t i = base + (int64_t)r * RS_BLOCK + threadIdx.x;
    if (i < n) h.count(keys[i], shift);
  }
  h.store(hist, tiles);
}

// Row scan: block d turns row d of the digit-major histogram (one count per tile) into exclusive
// offsets within the row and writes the row total to totals[d].
__global__ void __launch_bounds__(RS_BLOCK) k_radix_rowscan(uint32_t *__restrict__ hist, uint32_t tiles,
                                                            uint32_t *__restrict__ totals) {
  __shared__ uint32_t part[RS_WAVES];
  __shared__ uint32_t carry;
  int t = threadIdx.x;
  uint32_t *row = hist + (size_t)blockIdx.x * tiles;
  if (t == 0) carry = 0;
  __syncthreads();
  for (uint32_t base = 0; base < tiles; base += RS_BLOCK) {
    uint32_t i = base + t;
    uint32_t v = i < tiles ? row[i] : 0;
    uint32_t inc = wave_incl_scan(v);
    int w = t / WAVE, l = t % WAVE;
    if (l == WAVE - 1) part[w] = inc;
    __syncthreads();
    uint32_t off = carry;
    for (int k = 0; k < w; ++k) off += part[k];
    uint32_t excl = off + inc - v;
    if (i < tiles) row[i] = excl;
    __syncthreads();
    if (t == RS_BLOCK - 1) carry = excl + v;
    __syncthreads();
  }
  if (t == 0) totals[blockIdx.x] = carry;
}

// One tile of ITEMS * 256 pairs. Wave w takes the tile's w-th quarter, 64 consecutive pairs per
// round, so (wave, round, lane) is the input order and the sort stays stable. vin null: the values
// are the positions (first pass of an order). kout null: the keys are not needed any more.
template <int ITEMS>
__global__ void __launch_bounds__(RS_BLOCK) k_radix_scatter(const uint32_t *__restrict__ kin,
                                                            const uint32_t *__restrict__ vin,
                                                            uint32_t *__restrict__ kout, uint32_t *__restrict__ vout,
                                                            int64_t n, int shift, uint32_t tiles,
                                                            const uint32_t *__restrict__ offs,
                                                            const uint32_t *__restrict__ totals) {
  constexpr int TILE = RS_BLOCK * ITEMS;
  __shared__ uint32_t s_key[TILE], s_val[TILE];
  __shared__ volatile uint32_t s_cnt[RS_WAVES][256];
  __shared__ uint32_t s_goff[256];
  __shared__ uint32_t s_part[2][RS_WAVES];
  const int t = threadIdx.x, w = t / WAVE, lane = lane_id();
#pragma unroll
  for (int k = 0; k < RS_WAVES; ++k) s_cnt[k][t] = 0;
  const int64_t tile0 = (int64_t)blockIdx.x * TILE;
  const int count = (int)(n - tile0 < TILE ? n - tile0 : TILE);
  uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int j = w * (ITEMS * WAVE) + r * WAVE + lane;
    key[r] = j < count ? kin[tile0 + j] : 0u;
    val[r] = vin ? (j < count ? vin[tile0 + j] : 0u) : (uint32_t)(tile0 + j);
  }
  __syncthreads();
  const uint64_t lt = lanemask_lt();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int j = w * (ITEMS * WAVE) + r * WAVE + lane;
    const bool valid = j < count;
    const uint32_t d = (key[r] >> shift) & 0xFF;
    uint64_t peers = ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const uint64_t bb = ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? bb : ~bb;
    }
    const uint32_t before = (uint32_t)__popcll(peers & lt);
    const uint32_t c = s_cnt[w][d];
    rank[r] = c + before;
    __builtin_amdgcn_wave_barrier();
    if (valid && before == 0) s_cnt[w][d] = c + (uint32_t)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  {
    // thread t: digit t. Its first place in the tile (exclusive scan of the tile's counts), the
    // start of each wave's share of it, and the offset from tile places to output positions.
    uint32_t c[RS_WAVES], sum = 0;
#pragma unroll
    for (int k = 0; k < RS_WAVES; ++k) { c[k] = s_cnt[k][t]; sum += c[k]; }
    const uint32_t tot = totals[t];
    const uint32_t inc_l = wave_incl_scan(sum), inc_g = wave_incl_scan(tot);
    if (lane == WAVE - 1) { s_part[0][w] = inc_l; s_part[1][w] = inc_g; }
    __syncthreads();
    uint32_t lstart = inc_l - sum, gstart = inc_g - tot;
    for (int k = 0; k < w; ++k) { lstart += s_part[0][k]; gstart += s_part[1][k]; }
    uint32_t run = lstart;
#pragma unroll
    for (int k = 0; k < RS_WAVES; ++k) { s_cnt[k][t] = run; run += c[k]; }
    s_goff[t] = gstart + offs[(size_t)t * tiles + blockIdx.x] - lstart;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const int j = w * (ITEMS * WAVE) + r * WAVE + lane;
    if (j < count) {
      const uint32_t pos = s_cnt[w][(key[r] >> shift) & 0xFF] + rank[r];
      s_key[pos] = key[r];
      s_val[pos] = val[r];
    }
  }
  __syncthreads();
  for (int j = t; j < count; j += RS_BLOCK) {
    const uint32_t k = s_key[j];
    const uint32_t g = s_goff[(k >> shift) & 0xFF] + j;
    if (kout) kout[g] = k;
    vout[g] = s_val[j];
  }
}

RadixResult radix_sort_passes(uint32_t *keys, uint32_t *vals, uint32_t *tmp_keys, uint32_t *tmp_vals, uint32_t *hist,
                              int64_t n, int begin_bit, int end_bit, bool iota, bool want_keys, bool first_hist,
                              hipStream_t s) {
  const bool small = n <= RS_SMALL_MAX;
  const uint32_t tiles = ceil_div((uint64_t)n, small ? RS_TILE_SMALL : RS_TILE_LARGE);
  uint32_t *totals = hist + (size_t)256 * tiles;
  uint32_t *ka = keys, *va = vals, *kb = tmp_keys, *vb = tmp_vals;
  for (int shift = begin_bit; shift < end_bit; shift += 8) {
    const bool first = shift == begin_bit, last = shift + 8 >= end_bit;
    if (!(first && first_hist)) {
      if (small)
        hipLaunchKernelGGL(k_radix_hist<RS_ITEMS_SMALL>, dim3(tiles), dim3(RS_BLOCK), 0, s, ka, n, shift, tiles, hist);
      else
        hipLaunchKernelGGL(k_radix_hist<RS_ITEMS_LARGE>, dim3(tiles), dim3(RS_BLOCK), 0, s, ka, n, shift, tiles, hist);
      launch_check("k_radix_hist");
    }
    hipLaunchKernelGGL(k_radix_rowscan, dim3(256), dim3(RS_BLOCK), 0, s, hist, tiles, totals);
    launch_check("k_radix_rowscan");
    const uint32_t *vin = first && iota ? nullptr : va;
    uint32_t *kout = last && !want_keys ? nullptr : kb;
    if (small)
      hipLaunchKernelGGL(k_radix_scatter<RS_ITEMS_SMALL>, dim3(tiles), dim3(RS_BLOCK), 0, s, ka, vin, kout, vb, n,
                         shift, tiles, hist, totals);
    else
      hipLaunchKernelGGL(k_radix_scatter<RS_ITEMS_LARGE>, dim3(tiles), dim3(RS_BLOCK), 0, s, ka, vin, kout, vb, n,
                         shift, tiles, hist, totals);
    launch_check("k_radix_scatter");
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  return RadixResult{ka, va};
}

const uint32_t *radix_sort_order(uint32_t *keys, uint32_t *vals, uint32_t *tmp_keys, uint32_t *tmp_vals,
                                 uint32_t *hist, int64_t n, int begin_bit, int end_bit, bool first_hist,
                                 hipStream_t s) {
  return radix_sort_passes(keys, vals, tmp_keys, tmp_vals, hist, n, begin_bit, end_bit, true, false, first_hist, s)
      .vals;
}

void radix_sort_iota(uint32_t *keys, uint32_t *vals, uint32_t *tmp_keys, uint32_t *tmp_vals, uint32_t *hist,
                     int64_t n, int begin_bit, int end_bit, bool first_hist, hipStream_t s) {
  const RadixResult r =
      radix_sort_passes(keys, vals, tmp_keys, tmp_vals, hist, n, begin_bit, end_bit, true, true, first_hist, s);
  if (r.vals != vals) {
    THG_HIP(hipMemcpyAsync(keys, r.keys, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
    THG_HIP(hipMemcpyAsync(vals, r.vals, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
  }
}

}  // namespace thg
