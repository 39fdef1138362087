// Values to dim-major pages [blocks][nv][16] by runs of tokens (bf16).  A row's values are 2-byte stores 32 bytes apart, each into a line that other
// rows' workgroups write too, on other XCDs; they bound the kernels that write pages row by row.  A workgroup here takes the runs that begin in 16
// rows: neighbouring rows whose slots follow one another in a page.  A thread takes two values of all of a run's rows: it reads the rows in whole
// lines over the wave and writes a whole page's two values as 64 bytes, a part of a page's in 2-byte stores of its own.
// rotary_cache, 7830 rows of 2048 + 512 + 512 columns, 7168 apart, bf16: 51 -> 36 us together with its turning (25 of them without pages;
// the 112 MB take 20 at a copy's rate); qk_norm_cache, 8192 rows of 2048 + 512 + 512: 33 -> 26 (22 without pages).
// Not for rows of which each is another sequence's: runs of one row wait for the workgroup's others (294 rows of 16 + 2 heads of 64 4.0 us by rows, 7.7).
#pragma once
#include "hy_common.h"

namespace k8sllm {

constexpr int kValueRows = 16;       // rows whose runs a workgroup takes
constexpr long kValueRunRows = 256;  // steps of fewer rows write their values row by row: 300 rows 10.9 us by rows, 10.3 by runs

// base: the values' first column in row 0; part: of value_groups(), 512 columns of all rows after another
__device__ __forceinline__ void write_value_runs(const bf16_t* __restrict__ base, long stride, long rows, int part, int nv,
                                                 bf16_t* __restrict__ v_cache, const int* __restrict__ slots) {
  const int lane = threadIdx.x & 63, groups = (int)((rows + kValueRows - 1) / kValueRows);
  const long r0 = (long)(part % groups) * kValueRows;
  const int c = part / groups * 512 + 2 * threadIdx.x;
  // slots of rows r0 - 1 .. r0 + 62: a run has up to 16 rows and begins in the first 16
  const long rl = r0 - 1 + lane;
  const int sl = rl >= 0 && rl < rows ? slots[rl] : -1;
  const int before = __builtin_amdgcn_ds_bpermute(4 * max(lane - 1, 0), sl);
  const unsigned long long starts = __ballot(sl != before + 1 || (sl & 15) == 0 || before < 0);
  for (int i = 1; i <= kValueRows; ++i) {
    const int s0 = __builtin_amdgcn_readlane(sl, i);
    if (s0 < 0 || !(starts >> i & 1)) continue;
    const unsigned long long after = starts >> (i + 1);
    const int n = min(after ? __builtin_ctzll(after) + 1 : 16, 16 - (s0 & 15));
    const bf16_t* src = base + (r0 + i - 1) * stride;
    bf16_t* dst = v_cache + (long)(s0 >> 4) * nv * 16 + (s0 & 15);
    if (c < nv) {
      uint32_t v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j)  // past the run's end its last row again
        v[j] = *reinterpret_cast<const uint32_t*>(src + (uint32_t)(min(j, n - 1) * (int)stride + c));
      if (n == 16) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t lo = (v[2 * j] & 0xffffu) | (v[2 * j + 1] << 16);
          v[2 * j + 1] = (v[2 * j] >> 16) | (v[2 * j + 1] & 0xffff0000u);
          v[2 * j] = lo;
        }
        uint4* p = reinterpret_cast<uint4*>(dst + (uint32_t)(c * 16));
        p[0] = make_uint4(v[0], v[2], v[4], v[6]);
        p[1] = make_uint4(v[8], v[10], v[12], v[14]);
        p[2] = make_uint4(v[1], v[3], v[5], v[7]);
        p[3] = make_uint4(v[9], v[11], v[13], v[15]);
      } else {
        bf16_t* p = dst + (uint32_t)(c * 16);
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (j < n) {
            p[j] = (bf16_t)(v[j] & 0xffffu);
            p[16 + j] = (bf16_t)(v[j] >> 16);
          }
      }
    }
  }
}

// Workgroups that a step's values take
inline int value_groups(long rows, int nv) { return (int)((rows + kValueRows - 1) / kValueRows * ((nv + 511) / 512)); }

// What a launch needs for it: 16-token pages, two values a thread, pages on whole 16-byte pieces
inline bool value_runs_ok(const void* qkv, long stride, int v_col, int nv, const void* v_cache, const int* slots, long rows, int bs) {
  return rows >= kValueRunRows && v_cache != nullptr && slots != nullptr && bs == 16 && ((nv | v_col | stride) & 1) == 0 &&
         stride < (1l << 26) && nv < (1 << 26) &&
         (reinterpret_cast<uintptr_t>(qkv) & 3) == 0 && (reinterpret_cast<uintptr_t>(v_cache) & 15) == 0;
}

}  // namespace k8sllm
