// Shared device helpers and error plumbing for the atl HIP library (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>

namespace atlhip {

constexpr int kWave = 64;
constexpr int kBlock = 256;

// Last error message of this thread's most recent failing entry point (returned by atl_last_error()).
void set_error(const char* fmt, ...);

inline unsigned grid_for(int64_t n, int per_block = kBlock) {
  const int64_t g = (n + per_block - 1) / per_block;
  return (unsigned)(g < 1 ? 1 : g);
}

// Returns 0, or records the launch error and returns 1.
int check_launch(const char* what);

// ---------------------------------------------------------------------------------------------- device
// Order-preserving map of a float to a signed int (for atomic min/max of floats of any sign).
__device__ __forceinline__ int float_to_ordered(float f) {
  int i = __float_as_int(f);
  return i >= 0 ? i : i ^ 0x7fffffff;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, kWave);
  return v;
}

__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = max(v, __shfl_xor(v, d, kWave));
  return v;
}

__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = min(v, __shfl_xor(v, d, kWave));
  return v;
}

// A lane's value through a DPP row operation (gfx9: quad_perm, row mirrors, row_shr, row_bcast), no LDS permute.
template <int CTRL, int ROWS>
__device__ __forceinline__ float dppf(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xF, false));
}

// Sum over the 64 lanes, returned wave-uniform.
__device__ __forceinline__ float wave_sum_f(float v) {
  v += dppf<0xB1, 0xF>(v);                       // quad_perm [1, 0, 3, 2]
  v += dppf<0x4E, 0xF>(v);                       // quad_perm [2, 3, 0, 1]
  v += dppf<0x141, 0xF>(v);                      // row_half_mirror
  v += dppf<0x140, 0xF>(v);                      // row_mirror: every lane holds its row's sum
  v += dppf<0x142, 0xA>(v);                      // row_bcast:15 into rows 1, 3
  v += dppf<0x143, 0xC>(v);                      // row_bcast:31 into rows 2, 3: lane 63 holds the total
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// Lanes of a wave that are about to add to the same addresses (the same key) let one of them add their sums: global
// atomics on one cache line serialise (18 ns an event of four corners where all events meet in one pixel).  Up to
// kMergeRounds keys, each that of the first lane still open, are merged where at least kMergeMin lanes hold it; a key
// held by a tenth of the lanes is found with probability 1 - 0.9^8 = 0.57, and what it leaves is then spread over many
// waves.  Every lane of the wave calls it.  Returns whether this lane adds, with the sums in v.
constexpr int kMergeRounds = 8, kMergeMin = 4;
template <int NV>
__device__ __forceinline__ bool merge_lanes(bool live, int64_t key, float (&v)[NV]) {
  const int klo = (int)key, khi = (int)(key >> 32), lane = threadIdx.x & (kWave - 1);
  bool adds = live;
  uint64_t todo = __ballot(live);
  for (int r = 0; r < kMergeRounds && todo; ++r) {
    const int lead = __ffsll((unsigned long long)todo) - 1;
    const bool in = live && klo == __builtin_amdgcn_readlane(klo, lead) && khi == __builtin_amdgcn_readlane(khi, lead);
    const uint64_t same = __ballot(in);
    todo &= ~same;
    if (__popcll(same) < kMergeMin) continue;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const float s = wave_sum_f(in ? v[k] : 0.f);
      v[k] = in ? s : v[k];
    }
    adds = adds && (!in || lane == lead);
  }
  return adds;
}

// Exclusive scan of one int per thread over a block of BS threads.  `lds` holds BS/64 + 1 ints.
template <int BS>
__device__ __forceinline__ int block_exclusive_scan(int v, int* lds, int& total) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  int x = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int y = __shfl_up(x, d, kWave);
    if (lane >= d) x += y;
  }
  if (lane == kWave - 1) lds[wid] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int w = 0; w < BS / kWave; ++w) {
      const int t = lds[w];
      lds[w] = run;
      run += t;
    }
    lds[BS / kWave] = run;
  }
  __syncthreads();
  const int excl = x - v + lds[wid];
  total = lds[BS / kWave];
  __syncthreads();
  return excl;
}

}  // namespace atlhip
