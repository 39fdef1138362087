// Chunks of `len` rows numbered segment by segment: where chunk number c lies, and the number of a segment's first chunk.
// Every lane of a wave calls them together (they scan the segment table 64 entries at a time).
#pragma once
#include "hy_common.h"

namespace k8sllm {

constexpr int kChunk = 64;

struct ChunkAt {
  int seg, row, n;  // segment (-1: no such chunk), first row of the step, rows
  int k, count;     // the chunk's number within its segment, the segment's chunks
};

__device__ __forceinline__ ChunkAt chunk_at(const int* __restrict__ cu, int S, int c, int len = kChunk) {
  const int lane = threadIdx.x & 63;
  for (int b = 0; b < S; b += 64) {
    const int i = b + lane, r0 = i < S ? cu[i] : 0, n = i < S ? cu[i + 1] - r0 : 0, nt = (n + len - 1) / len;
    int incl = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(incl, o, 64);
      if (lane >= o) incl += up;
    }
    const unsigned long long past = __ballot(incl > c);
    if (past != 0) {
      const int f = __builtin_ctzll(past);
      const int k = c - (__shfl(incl, f, 64) - __shfl(nt, f, 64)), rows = __shfl(n, f, 64);
      return {__builtin_amdgcn_readfirstlane(b + f), __builtin_amdgcn_readfirstlane(__shfl(r0, f, 64) + k * len),
              __builtin_amdgcn_readfirstlane(min(len, rows - k * len)), __builtin_amdgcn_readfirstlane(k),
              __builtin_amdgcn_readfirstlane(__shfl(nt, f, 64))};
    }
    c -= __shfl(incl, 63, 64);
  }
  return {-1, 0, 0, 0, 0};
}

__device__ __forceinline__ int first_chunk(const int* __restrict__ cu, int s) {
  const int lane = threadIdx.x & 63;
  int total = 0;
  for (int b = 0; b < s; b += 64) {
    const int i = b + lane, n = i < s ? cu[i + 1] - cu[i] : 0;
    total += (int)wave_sum_dpp((float)((n + kChunk - 1) / kChunk));  // exact: fewer than 2^24 chunks
  }
  return __builtin_amdgcn_readfirstlane(total);
}

}  // namespace k8sllm
