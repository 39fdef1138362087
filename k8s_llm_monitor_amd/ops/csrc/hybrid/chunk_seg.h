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

// Which segment the r-th group of ``per`` workgroups takes.  The longest ones first, one workgroup a unit, then those that come beside them from the
// shortest on, and so on: workgroups go to the units in turn, and a chain of tokens beside another takes up to twice as long, so that a step of
// prompts of different lengths took as long as its two longest ones on one unit.  us, in the step's order / so: 13 prompts of 45 to 901 tokens, selective
// scan of 2048 channels 150 / 123, delta rule of 8 heads 110 / 104, linear attention of 16 85 / 75, wkv of 16 87 / 84; 32 such prompts, linear attention of
// 8 108 / 87.  No more workgroups than units, more than ``most`` of them or more than 64 segments: from the last one on (a step's prompts come after its
// running sequences).  Short segments behind one another pay for the choice (64 of 5 to 94 tokens, delta rule of 8 heads 93 / 104, linear attention of 16
// 59 / 67), and over many rounds they even out by themselves (64 of 45 to 901 tokens, delta rule of 16 heads 811 / 812), so the chunks' scans make none
// beyond four rounds; the selective scan, whose tokens take longest, does (64 of 5 to 94 tokens, 4096 channels 103 / 69, of 45 to 901 880 / 535).  Equal
// lengths cost nothing or 1 us (64 of 64 tokens, linear attention of 8 heads 31.0 / 31.4; 16 of 500 42 / 42).
// The lanes hold the whole table, so that nothing is loaded behind the choice; the r-th longest is found from the highest bit of the lengths on.
struct SegAt {
  int seg, slot, t0, t1;  // its rows: t0 .. t1 - 1
};
__device__ __forceinline__ SegAt segment_in_turn(const int* __restrict__ cu, const int* __restrict__ slot, int S, int r, int per,
                                                 int most = 1024) {
  if (S * per <= 256 || S * per > most || S > 64) {
    const int s = S - 1 - r;
    return {s, slot[s], cu[s], cu[s + 1]};
  }
  const int round = max(1, 256 / per);
  const int lane = threadIdx.x & 63, i = min(lane, S - 1), c = cu[i], n = cu[i + 1] - c, sl = slot[i], k = r / round;
  if (k & 1) r = min((k + 1) * round, S) - 1 - (r - k * round);
  // those that may be the r-th longest (of equal ones in the step's order)
  unsigned long long left = S == 64 ? ~0ull : (1ull << S) - 1;
  if (__ballot(n != __builtin_amdgcn_readfirstlane(n)) != 0)
    for (int bit = __ballot(n >> 12) ? 30 : 11; bit >= 0 && (left & (left - 1)); --bit) {
      const unsigned long long on = left & __ballot((n >> bit) & 1);
      const int more = __popcll(on);
      if (r < more) {
        left = on;
      } else {
        r -= more;
        left &= ~on;
      }
    }
  const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(left >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)left, 0));
  const int s = __builtin_ctzll(__ballot(before == r) & left), t0 = __builtin_amdgcn_readlane(c, s);
  return {s, __builtin_amdgcn_readlane(sl, s), t0, t0 + __builtin_amdgcn_readlane(n, s)};
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
