// The first pass of the permute (permute.hip), shared with the prefill's prep kernel.
#pragma once

#include "wm_common.h"

namespace wm {

constexpr int PERMUTE_CHUNK = 256;
constexpr int PERMUTE_MAX_EXPERTS = 1024;
constexpr int PERMUTE_COUNT_WAVES = 4;  // chunks a block

// Chunks of pairs counted by block `block`, one a wave; block 0 also clears the counter `done` of the
// scan after it. Every thread of the block calls it.
__device__ __forceinline__ void permute_count_block(const int32_t* __restrict__ idx, int64_t pairs, int experts,
                                                    int64_t block, int32_t* __restrict__ chunk_counts,
                                                    int32_t* __restrict__ done) {
  __shared__ int32_t all_counts[PERMUTE_COUNT_WAVES][PERMUTE_MAX_EXPERTS];
  int32_t* counts = all_counts[threadIdx.x / 64];
  const int lane = threadIdx.x % 64;
  const int64_t chunks = (pairs + PERMUTE_CHUNK - 1) / PERMUTE_CHUNK;
  const int64_t chunk = block * PERMUTE_COUNT_WAVES + threadIdx.x / 64;
  if (block == 0 && threadIdx.x == 0) *done = 0;
  for (int e = lane; e < experts; e += 64) counts[e] = 0;
  __syncthreads();
  const int64_t begin = chunk * PERMUTE_CHUNK, end = min<int64_t>(pairs, begin + PERMUTE_CHUNK);
  for (int64_t p = begin + lane; p < end; p += 64) {
    const int e = idx[p];
    if (e >= 0 && e < experts) atomicAdd(&counts[e], 1);
  }
  __syncthreads();
  if (chunk < chunks)
    for (int e = lane; e < experts; e += 64) chunk_counts[chunk * experts + e] = counts[e];
}

// Blocks of permute_count_block for a list of pairs.
inline int64_t permute_count_blocks(int64_t pairs) {
  const int64_t n = (pairs + PERMUTE_CHUNK * PERMUTE_COUNT_WAVES - 1) / (PERMUTE_CHUNK * PERMUTE_COUNT_WAVES);
  return n > 0 ? n : 1;
}

}  // namespace wm
