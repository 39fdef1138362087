// Helpers shared by the layer-list decoders' kernels: activations are either bf16 (raw 16-bit
// patterns, common.h) or fp32, selected by a template parameter; all arithmetic is fp32.
#pragma once
#include "common.h"

namespace k8sllm {

template <typename T>
__device__ __forceinline__ float ldf(const T* p);
template <>
__device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float ldf<bf16_t>(const bf16_t* p) { return bf2f(*p); }

template <typename T>
__device__ __forceinline__ void stf(T* p, float v);
template <>
__device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void stf<bf16_t>(bf16_t* p, float v) { *p = f2bf(v); }

// element i of a tensor whose dtype is only known at run time: 1 = bf16, 2 = fp32
__device__ __forceinline__ float ld_any(const void* p, int dt, long i) {
  return dt == 2 ? reinterpret_cast<const float*>(p)[i] : bf2f(reinterpret_cast<const bf16_t*>(p)[i]);
}

// 8 consecutive elements (16-byte aligned for bf16, 32-byte for fp32) as floats, and back
__device__ __forceinline__ void load8(const bf16_t* p, float* f) { unpack8(*reinterpret_cast<const uint4*>(p), f); }
__device__ __forceinline__ void load8(const float* p, float* f) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
  f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}
// 4 consecutive elements (8-byte aligned for bf16, 16-byte for fp32)
__device__ __forceinline__ void load4(const bf16_t* p, float* f) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
}
__device__ __forceinline__ void load4(const float* p, float* f) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
}
__device__ __forceinline__ void store8(bf16_t* p, const float* f) { *reinterpret_cast<uint4*>(p) = pack8(f); }
__device__ __forceinline__ void store8(float* p, const float* f) {
  *reinterpret_cast<float4*>(p) = make_float4(f[0], f[1], f[2], f[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(f[4], f[5], f[6], f[7]);
}
__device__ __forceinline__ void load8_any(const void* p, int dt, long i, float* f) {
  if (dt == 2) load8(reinterpret_cast<const float*>(p) + i, f);
  else load8(reinterpret_cast<const bf16_t*>(p) + i, f);
}

// Four fp32 of a recurrent state; ONCE: non-temporal, where a step's states are more than the caches keep until the next step
constexpr long kStateOnceBytes = 8l << 20;
using f32v4 = float __attribute__((ext_vector_type(4)));
template <bool ONCE>
__device__ __forceinline__ f32v4 load_state(const float* p) {
  const f32v4* q = reinterpret_cast<const f32v4*>(p);
  return ONCE ? __builtin_nontemporal_load(q) : *q;
}
template <bool ONCE>
__device__ __forceinline__ void store_state(float* p, f32v4 v) {
  f32v4* q = reinterpret_cast<f32v4*>(p);
  if (ONCE) __builtin_nontemporal_store(v, q);
  else *q = v;
}

// Eight 16-bit values of tokens j .. j + 7, zero where not (j < end): what lies behind a sequence's last token in its last page is
// another sequence's, and a weight of zero does not take away a NaN
__device__ __forceinline__ uint32_t pair_below(int j, int end) { return j + 1 < end ? ~0u : j < end ? 0xffffu : 0u; }
__device__ __forceinline__ uint4 tokens_below(uint4 v, int j, int end) {
  return make_uint4(v.x & pair_below(j, end), v.y & pair_below(j + 2, end), v.z & pair_below(j + 4, end), v.w & pair_below(j + 6, end));
}

// Two values' sums at once: even rows (the lower half) end with a's sum over the two rows (halves), odd ones (the upper) with b's
__device__ __forceinline__ float swap16_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap32_sum(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// as wave_sum and wave_max, nearest lanes first
__device__ __forceinline__ float wave_sum_dpp(float v) {
  v += K8SLLM_DPP(v, 0xB1);
  v += K8SLLM_DPP(v, 0x4E);
  v += K8SLLM_DPP(v, 0x141);
  v += K8SLLM_DPP(v, 0x140);
  return xor32_sum_f(xor16_sum(v));
}
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = fmaxf(v, K8SLLM_DPP(v, 0xB1));
  v = fmaxf(v, K8SLLM_DPP(v, 0x4E));
  v = fmaxf(v, K8SLLM_DPP(v, 0x141));
  v = fmaxf(v, K8SLLM_DPP(v, 0x140));
  return xor32_max_f(xor16_max(v));
}

__device__ __forceinline__ float silu_f(float z) { return z / (1.f + __expf(-z)); }
__device__ __forceinline__ float sigmoid_f(float z) { return 1.f / (1.f + expf(-z)); }

// four rounded values times the sigmoids of their logits, rounded again
__device__ __forceinline__ uint2 gate_rounded(uint2 x, uint2 z) {
  auto half = [](uint32_t a, uint32_t b) {
    return pack2(__uint_as_float(a << 16) * sigmoid_f(__uint_as_float(b << 16)),
                 __uint_as_float(a & 0xffff0000u) * sigmoid_f(__uint_as_float(b & 0xffff0000u)));
  };
  return make_uint2(half(x.x, z.x), half(x.y, z.y));
}

// Where row tile ``tile`` of ROWS rows lies among experts whose rows are offsets[e] .. offsets[e + 1] - 1: expert e, its rows r0 .. r1 - 1 and the
// tile's number in it; false behind the last.  Up to 64 experts one after another, from the scalar cache; more of them 64 at a time, a
// lane each (the sum over 64 takes about 1 us, of a load that waits behind the weights': 2 rows beside 128 experts 46 -> 13 us, 64 rows
// beside 64 24.6 -> 25.9).
template <int ROWS>
__device__ __forceinline__ bool expert_tile(const int* __restrict__ offsets, int E, int& tile, int& e, int& r0, int& r1) {
  if (E <= 64) {
    for (e = 0; e < E; ++e) {
      r0 = offsets[e];
      r1 = offsets[e + 1];
      const int n = (r1 - r0 + ROWS - 1) / ROWS;
      if (tile < n) return true;
      tile -= n;
    }
    return false;
  }
  const int lane = threadIdx.x & 63;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int i = min(e0 + lane, E - 1), a = offsets[i], b = offsets[i + 1], n = e0 + lane < E ? (b - a + ROWS - 1) / ROWS : 0;
    int s = n;  // sums up to this lane: in rows of 16 lanes, then over the rows
    s += __builtin_amdgcn_update_dpp(0, s, 0x111, 0xf, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x112, 0xf, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x114, 0xf, 0xf, true);
    s += __builtin_amdgcn_update_dpp(0, s, 0x118, 0xf, 0xf, true);
    const int s0 = __builtin_amdgcn_readlane(s, 15), s1 = s0 + __builtin_amdgcn_readlane(s, 31), s2 = s1 + __builtin_amdgcn_readlane(s, 47);
    const int all = s2 + __builtin_amdgcn_readlane(s, 63);
    s += lane < 16 ? 0 : lane < 32 ? s0 : lane < 48 ? s1 : s2;
    if (tile < all) {
      const int l = __builtin_ctzll(__ballot(s > tile));
      e = e0 + l;
      r0 = __builtin_amdgcn_readlane(a, l);
      r1 = __builtin_amdgcn_readlane(b, l);
      tile -= __builtin_amdgcn_readlane(s - n, l);
      return true;
    }
    tile -= all;
  }
  return false;
}

// KIND 0: erf GELU, 1: tanh GELU, 2: xIELU (a z^2 + z/2 above zero, b (exp(z) - 1 - z) + z/2 below), 3: SiLU,
// 4: ReLU, 6: squared ReLU, 7: tanh (5 is a gated unit, glu_unit)
template <int KIND>
__device__ __forceinline__ float act_f(float z, float a, float b) {
  if (KIND == 6) return z > 0.f ? z * z : 0.f;
  if (KIND == 7) return tanhf(z);
  if (KIND == 4) return fmaxf(z, 0.f);
  if (KIND == 0) return 0.5f * z * (1.f + erff(z * 0.70710678118654752f));
  if (KIND == 1) return 0.5f * z * (1.f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)));
  if (KIND == 3) return z / (1.f + expf(-z));
  return z > 0.f ? a * z * z + 0.5f * z : b * (expm1f(z) - z) + 0.5f * z;
}

// KIND 5: the clamped unit g sigmoid(1.702 g) (u + 1) with g = min(gate, limit), u = clamp(up, -limit, limit);
// others: act(gate) * up
template <int KIND>
__device__ __forceinline__ float glu_unit(float g, float u, float limit) {
  if (KIND == 5) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g * sigmoid_f(1.702f * g) * (u + 1.f);
  }
  return act_f<KIND>(g, 0.f, 0.f) * u;
}

// sum over groups of CH neighbouring lanes (CH a power of two <= 32, groups aligned); every lane of a group
// ends with its total
template <int CH>
__device__ __forceinline__ float lanes_sum(float v) {
  if (CH >= 2) v += K8SLLM_DPP(v, 0xB1);
  if (CH >= 4) v += K8SLLM_DPP(v, 0x4E);
  if (CH >= 8) v += K8SLLM_DPP(v, 0x141);
  if (CH >= 16) v += K8SLLM_DPP(v, 0x140);
  if (CH >= 32) v = xor16_sum(v);
  return v;
}

__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// windowed attention: the first position that a row at position p sees
__device__ __forceinline__ int first_key(int p, int window, int chunked) {
  if (window <= 0) return 0;
  return chunked ? p - p % window : max(0, p - window + 1);
}

// the segment that holds row r: largest s with cu[s] <= r (cu has S + 1 entries, cu[0] = 0)
__device__ __forceinline__ int find_segment(const int* __restrict__ cu, int S, int r) {
  int lo = 0, hi = S - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= r) lo = mid; else hi = mid - 1;
  }
  return lo;
}

}  // namespace k8sllm
