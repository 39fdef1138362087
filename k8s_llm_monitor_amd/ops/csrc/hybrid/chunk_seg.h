// Chunks of `len` rows numbered segment by segment: where chunk number c lies, and the number of a segment's first chunk.
// Every lane of a wave calls them together (they scan the segment table 64 entries at a time).
#pragma once
#include "hy_common.h"

namespace k8sllm {

constexpr int kChunk = 64;

// The chunked recurrences multiply the values of a chunk by weights that are zero for the tokens in front of them.  So that an
// infinity or NaN reaches no earlier token, as token by token, such a value is staged as zero, the first row at which it stood in a
// column is kept (kNone: there was none), and the column's results are NaN from that row on, its state with them.
constexpr int kNone = kChunk;
__device__ __forceinline__ bool odd_bf16(uint32_t x) { return (x & 0x7f80u) == 0x7f80u; }  // infinity or NaN
__device__ __forceinline__ bool odd_pair(uint32_t w) { return odd_bf16(w) || odd_bf16(w >> 16); }
// stages VW bf16 values of row `row` of n (words w) as above; first: their columns' first rows
template <int VW>
__device__ __forceinline__ void keep_finite(uint32_t (&w)[VW / 2], int row, int n, int* first) {
  bool any = false;
#pragma unroll
  for (int i = 0; i < VW / 2; ++i) any |= odd_pair(w[i]);
  if (!any) return;
#pragma unroll
  for (int i = 0; i < VW; ++i)
    if (odd_bf16(w[i / 2] >> (16 * (i & 1)))) {
      w[i / 2] &= i & 1 ? 0x0000ffffu : 0xffff0000u;
      if (row < n) atomicMin(first + i, row);
    }
}

// log2 of a decay from its logit (kinds of decay_scan.hip); 2^-4096 is zero in fp32, and a NaN stays one
__device__ __forceinline__ float log2_decay(float x, int kind, float A, float inv_tau) {
  auto softplus = [](float v) {  // softplus_f without a branch, so that a run of tokens is evaluated side by side
    const float r = log1pf(expf(v > 20.f ? 20.f : v));
    return v > 20.f ? v : r;
  };
  const float e = kind == 0 ? A * softplus(x) : kind == 1 ? softplus(-x) * inv_tau : expf(x);
  const float l = -1.44269504088896341f * e;
  return l < -4096.f ? -4096.f : l;
}

// what a workgroup of a scan owns: a whole segment, or one of the spans that a long one is cut into - the launch that leaves the
// spans' end states, and the one that folds those in front of its own
constexpr int kWhole = 0, kSpanEnds = 1, kSpanRun = 2;

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

// Which segment the r-th group of workgroups takes, where one workgroup a compute unit is `round` groups: the longest ones first, one a unit, then
// the shortest first, which come beside them (workgroups go to the units in turn), and so on.  A chain of tokens beside another takes up to twice as
// long, so that a step of prompts of different lengths took as long as its two longest ones on one unit: 13 prompts of 45 to 901 tokens, us, in the
// step's order / so: selective scan of 2048 channels 144 / 126, delta rule of 8 heads 72 / 58, wkv of 16 50 / 43.  More than 64 segments: from
// the last one on (a step's prompts come after its running sequences).
__device__ __forceinline__ int segment_in_turn(const int* __restrict__ cu, int S, int r, int round) {
  if (S <= 1 || S > 64) return S - 1 - r;
  const int k = r / round;
  if (k & 1) r = min((k + 1) * round, S) - 1 - (r - k * round);
  const int lane = threadIdx.x & 63, n = lane < S ? cu[lane + 1] - cu[lane] : -1;
  int rank = 0;
  for (int j = 0; j < S; ++j) {
    const int m = __builtin_amdgcn_readlane(n, j);
    rank += m > n || (m == n && j < lane);
  }
  return __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(lane < S && rank == r)));
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
