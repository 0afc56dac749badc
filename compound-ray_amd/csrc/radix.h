// Stable LSD radix sort passes (8 bits each) of (key, uint32 value) pairs, keys
// of 32 or 64 bits; a pass is k_sort_hist, an exclusive scan of the histogram
// (scan.h) and k_sort_scatter.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace eye {
namespace {

constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr int kRadix = 256;
constexpr int kWaves = kSortThreads / 64;

// Per-tile digit histogram, written digit-major: hist[digit * tiles + tile].
template <typename K>
__global__ __launch_bounds__(kSortThreads) void k_sort_hist(const K* __restrict__ keys, int n,
                                                            int shift, uint32_t* __restrict__ hist,
                                                            int tiles) {
  __shared__ uint32_t h[kRadix];
  h[threadIdx.x] = 0;
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * kSortTile;
  for (int j = 0; j < kSortItems; ++j) {
    const size_t idx = base + (size_t)j * kSortThreads + threadIdx.x;
    if (idx < (size_t)n) atomicAdd(&h[(uint32_t)(keys[idx] >> shift) & (kRadix - 1)], 1u);
  }
  __syncthreads();
  hist[(size_t)threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter.  Items are taken in the order (item j, wave, lane); ranks
// among equal digits inside a wave come from ballot matching, across waves
// and items from LDS running counters, across tiles from the scanned
// histogram.
template <typename K>
__global__ __launch_bounds__(kSortThreads) void k_sort_scatter(
    const K* __restrict__ kin, const uint32_t* __restrict__ vin, K* __restrict__ kout,
    uint32_t* __restrict__ vout, int n, int shift, const uint32_t* __restrict__ offs, int tiles) {
  __shared__ uint32_t wave_cnt[kWaves][kRadix];
  __shared__ uint32_t wave_off[kWaves][kRadix];
  __shared__ uint32_t run_base[kRadix];
  __shared__ uint32_t g_off[kRadix];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  run_base[tid] = 0;
  g_off[tid] = offs[(size_t)tid * tiles + blockIdx.x];
  const uint64_t lt_mask = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
  const size_t base = (size_t)blockIdx.x * kSortTile;
  for (int j = 0; j < kSortItems; ++j) {
    const size_t idx = base + (size_t)j * kSortThreads + tid;
    const bool valid = idx < (size_t)n;
    const K key = valid ? kin[idx] : (K)0;
    const uint32_t val = valid ? vin[idx] : 0u;
    const uint32_t d = (uint32_t)(key >> shift) & (kRadix - 1);
    for (int k = 0; k < kWaves; ++k) wave_cnt[k][tid] = 0;
    __syncthreads();
    uint64_t peers = __ballot(valid);
    for (int b = 0; b < 8; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    uint32_t rank = 0;
    if (valid) {
      rank = (uint32_t)__popcll(peers & lt_mask);
      const int leader = 63 - __clzll((long long)peers);
      if (leader == lane) wave_cnt[w][d] = (uint32_t)__popcll(peers);
    }
    __syncthreads();
    {
      uint32_t run = run_base[tid];
      for (int k = 0; k < kWaves; ++k) {
        const uint32_t c = wave_cnt[k][tid];
        wave_off[k][tid] = run;
        run += c;
      }
      run_base[tid] = run;
    }
    __syncthreads();
    if (valid) {
      const uint32_t pos = g_off[d] + wave_off[w][d] + rank;
      if (pos < (uint32_t)n) {  // always true for a consistent histogram; never write out of bounds
        kout[pos] = key;
        vout[pos] = val;
      }
    }
  }
}

}  // namespace
}  // namespace eye
