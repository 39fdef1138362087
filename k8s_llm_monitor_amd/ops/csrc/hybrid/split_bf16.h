// fp32 operands on the bf16 matrix instructions without losing bits: an fp32 number is the sum of three bf16 numbers
// (truncation takes 8 mantissa bits each time, and the differences are exact), bf16 products are exact in the
// instruction's fp32 accumulator, so (fp32 a) x (bf16 b) as three instructions rounds only where the fp32 sums do.  At a
// sixteenth of the bf16 rate for the fp32 instruction that is about five times as fast.
#pragma once
#include "hy_common.h"

namespace k8sllm {

typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ __forceinline__ void split3(float x, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = __float_as_uint(x) & 0xffff0000u;
  const float r = x - __uint_as_float(h);
  m = __float_as_uint(r) & 0xffff0000u;
  l = __float_as_uint(r - __uint_as_float(m));
}
// the bf16 patterns in the upper halves of a and b as one word, a first
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302); }

// 2 N fp32 values as three packed rows of bf16 pairs
template <int N>
__device__ __forceinline__ void split_pairs(const float* x, uint32_t* h, uint32_t* m, uint32_t* l) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    uint32_t ha, ma, la, hb, mb, lb;
    split3(x[2 * i], ha, ma, la);
    split3(x[2 * i + 1], hb, mb, lb);
    h[i] = pack_hi(ha, hb);
    m[i] = pack_hi(ma, mb);
    l[i] = pack_hi(la, lb);
  }
}

__device__ __forceinline__ bf16x8 frag(const uint32_t* w) {
  return __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}

// A workgroup barrier for data that passes through LDS: unlike __syncthreads() it leaves global loads in flight (a
// prefetch across the barrier) instead of waiting for them.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// An operand fragment whose k index runs down the rows of a row-major LDS matrix (row pitch in elements): this lane's
// column c0 + (lane & 15), rows r0 .. r0 + 3 and r1 .. r1 + 3.  The transposing read takes, for 16 lanes, four rows of 16
// columns and gives each lane one column's four rows.
__device__ __forceinline__ bf16x8 frag_down(const bf16_t* m, int pitch, int r0, int r1, int c0) {
  const int i = threadIdx.x & 15;
  const bf16_t* p = m + (i >> 2) * pitch + c0 + 4 * (i & 3);
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + r0 * pitch));
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + r1 * pitch));
  const uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
  return __builtin_bit_cast(bf16x8, make_uint4(x.x, x.y, y.x, y.y));
}

}  // namespace k8sllm
