// Device helpers shared by the kernel files: wave-level primitives, ordered-float atomics,
// XCD-aware block remapping, launch checking.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"

namespace thg {

constexpr int WAVE = 64;  // CDNA wavefront width

__device__ __forceinline__ int lane_id() { return __lane_id(); }
// Wave-wide ballot of a lane predicate straight from the compare mask (no 0/1 round trip).
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

__device__ __forceinline__ uint64_t lanemask_lt() {
  int l = lane_id();
  return l == 0 ? 0ull : (~0ull >> (64 - l));
}

// Order-preserving float <-> int maps for integer atomicMin/atomicMax on floats.
__device__ __forceinline__ int float_to_ord(float f) {
  int i = __float_as_int(f);
  return i >= 0 ? i : i ^ 0x7fffffff;
}
__host__ __device__ __forceinline__ float ord_to_float(int i) {
  int j = i >= 0 ? i : i ^ 0x7fffffff;
  union { int i; float f; } u;
  u.i = j;
  return u.f;
}

template <typename T> __device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, WAVE);
  return v;
}
__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fminf(v, __shfl_xor(v, off, WAVE));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, WAVE));
  return v;
}

// Inclusive scan across the wave.
template <typename T> __device__ __forceinline__ T wave_incl_scan(T v) {
  int l = lane_id();
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    T o = __shfl_up(v, off, WAVE);
    if (l >= off) v += o;
  }
  return v;
}

// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD b % 8). Remap so the
// blocks an XCD runs cover one contiguous range of logical blocks: neighbouring (spatially sorted)
// work then shares that XCD's L2. `nb` must be a multiple of 8; logical ids >= the real block count
// are skipped by the caller.
__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t nb) {
  const uint32_t X = 8;
  uint32_t per = nb / X;
  return (b % X) * per + b / X;
}

inline uint32_t round_up8(uint64_t nb) { return (uint32_t)((nb + 7) / 8 * 8); }

// A pointer read from a descriptor in device memory reaches the compiler as a generic (flat)
// pointer, and loads through it go to the vector memory path even when every lane reads the same
// address. The trees, records and queries a traversal reads are device memory that no wave writes
// while the kernel runs: reading the descriptor's field as a pointer to the constant address space
// (device memory that is read-only for the kernel's duration) lets the compiler carry that into the
// inlined traversal, so its wave-uniform node and record loads become scalar loads, as they are when
// the same pointers arrive as const __restrict__ kernel arguments. Loads that differ across lanes
// stay vector loads.
template <typename T, typename F> __device__ __forceinline__ const T *readonly_ptr(F *const &field) {
  typedef const __attribute__((address_space(4))) T *cptr;
  return (const T *)*reinterpret_cast<const cptr *>(reinterpret_cast<const void *>(&field));
}

inline void launch_check(const char *name) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) fail(THG_E_DEVICE, std::string("kernel launch ") + name + ": " + hipGetErrorString(e));
}

inline uint32_t ceil_div(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// Radix sort (radix_sort.hip): 8-bit digits, tiles of 1,024 pairs up to 2^20 pairs (a tile of 4,096
// would leave most CUs idle: 25 workgroups for 100,000 pairs) and of 4,096 above (runs of equal
// digits four times as long to write).
constexpr int RS_BLOCK = 256;
constexpr int RS_ITEMS_SMALL = 4, RS_ITEMS_LARGE = 16;
constexpr uint64_t RS_TILE_SMALL = RS_BLOCK * RS_ITEMS_SMALL, RS_TILE_LARGE = RS_BLOCK * RS_ITEMS_LARGE;
constexpr int64_t RS_SMALL_MAX = (int64_t)1 << 20;

// Digit counts of one tile, in LDS. A key kernel that processes whole tiles in 256-thread blocks
// fills one (clear, count every key, store) and so saves the sort its first histogram pass.
struct RadixHist {
  uint32_t h[256];
  __device__ __forceinline__ void clear() {
    h[threadIdx.x] = 0;
    __syncthreads();
  }
  __device__ __forceinline__ void count(uint32_t key, int shift) { atomicAdd(&h[(key >> shift) & 0xFF], 1u); }
  __device__ __forceinline__ void store(uint32_t *__restrict__ hist, uint32_t tiles) {
    __syncthreads();
    hist[(size_t)threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
  }
};
inline int radix_items(int64_t n) { return n <= RS_SMALL_MAX ? RS_ITEMS_SMALL : RS_ITEMS_LARGE; }
inline uint32_t radix_tiles(int64_t n) { return ceil_div((uint64_t)n, (uint64_t)RS_BLOCK * radix_items(n)); }

// Where a sort left its results.
struct RadixResult {
  const uint32_t *keys, *vals;
};

// The stable order of n keys by bits [begin_bit, end_bit): returns the positions in that order, in
// vals or tmp_vals. vals needs no input; the keys' own order is lost. first_hist: the caller's key
// kernel has stored the first digit's histograms (RadixHist) in hist. `hist` must hold
// radix_hist_words(n) words.
const uint32_t *radix_sort_order(uint32_t *keys, uint32_t *vals, uint32_t *tmp_keys, uint32_t *tmp_vals,
                                 uint32_t *hist, int64_t n, int begin_bit, int end_bit, bool first_hist,
                                 hipStream_t s);
// The same order with the sorted keys in `keys` and the positions in `vals`.
void radix_sort_iota(uint32_t *keys, uint32_t *vals, uint32_t *tmp_keys, uint32_t *tmp_vals, uint32_t *hist,
                     int64_t n, int begin_bit, int end_bit, bool first_hist, hipStream_t s);
size_t radix_hist_words(int64_t n);

}  // namespace thg
