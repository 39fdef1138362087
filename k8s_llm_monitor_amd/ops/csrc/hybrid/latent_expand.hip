// Per-head keys and values of latent attention, expanded from the latent pages into temporary pages that the windowed
// attention kernels read: for every listed latent page [16][pitch] (rows [latent c of R | shared key part of dr | ...])
//   keys   [page][16][H * (dn + dr)]   per head [W_uk[h] c | shared part]
//   values [page][H][dv][16]           W_uv[h] c
// in bf16 with fp32 sums, one rounding.  R 128 or 256, dn and dv multiples of 32, dr a multiple of 8.
//
// What bounds it: writing 2 (dn + dr + dv) H bytes per token.  A workgroup of four waves takes 128 tokens (8 pages, found
// through the page list: no gathered copy of the latents) and one head; a wave keeps its 32 tokens' latents in
// registers as matrix operands for the whole launch, the head's weight rows pass through LDS in tiles of 32 x R, copied
// there by global_load_lds (two tiles in flight, pieces of 16 bytes swizzled by row).  The keys' product has the dims on the
// accumulator rows and the values' the tokens, each in the order that swaps bits 2 and 3 of the row number: a lane then
// holds 8 consecutive dims of one token (keys) or 8 consecutive tokens of one dim (values), one 16-byte store; the
// value pages are written 1 KiB contiguous per store instruction, already dim-major.
// Measured, 16 heads, 96 + 32 / 128 dims, R 256: 8000 tokens 42 us (65 MB written, 14.7 GFLOP), where the matrix products, the
// copies around them, the zero fills and the page-writing pass that this kernel replaces took 260 us.
#include "hy_common.h"

namespace k8sllm {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void gbl_void_t;

template <int R>
__global__ __launch_bounds__(256) void latent_expand_kernel(bf16_t* __restrict__ kt, bf16_t* __restrict__ vt,
                                                            const bf16_t* __restrict__ k_cache, int pitch,
                                                            const int* __restrict__ page_list, int npages,
                                                            const bf16_t* __restrict__ wk, const bf16_t* __restrict__ wv,
                                                            int H, int dn, int dr, int dv) {
  constexpr int KS = R / 16, CH = R / 8, TILE = 32 * R * 2, NP = TILE / 4096;  // NP: 1 KiB copies per wave and tile
  __shared__ __attribute__((aligned(16))) char ring[2 * TILE];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r32 = lane & 31, hh = lane >> 5, h = blockIdx.x;
  const int perm = (r32 & ~12) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);
  const int D = dn + dr;
  const int p0 = blockIdx.y * 8 + wave * 2;  // this wave's two pages (index into the list)
  const int nk = dn / 32, nt = nk + dv / 32;
  auto issue = [&](int t, int slot) {
    const bf16_t* w = t < nk ? wk + ((long)h * dn + 32 * t) * R : wv + ((long)h * dv + 32 * (t - nk)) * R;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int c = (wave * NP + i) * 64 + lane, row = c / CH, ch = (c % CH) ^ (row & 15);
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(w + row * R + ch * 8), (lds_void_t*)(ring + slot * TILE + (wave * NP + i) * 1024),
                                       16, 0, 0);
    }
  };
  // the wave's latents: token r32 in list order for the keys (lane = token), and in swapped order for the values, whose
  // accumulator rows are tokens
  auto src = [&](int tok) {
    const long page = page_list[min(p0 + (tok >> 4), npages - 1)];
    return k_cache + (page * 16 + (tok & 15)) * pitch;
  };
  bf16x8 ck[KS], cv[KS];
  {
    const bf16_t *a = src(r32), *b = src(perm);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ck[ks] = *reinterpret_cast<const bf16x8*>(a + 16 * ks + 8 * hh);
      cv[ks] = *reinterpret_cast<const bf16x8*>(b + 16 * ks + 8 * hh);
    }
  }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(ck[ks]), "v"(cv[ks]));  // waited for before the copies start
  auto half = [](const f32x16& a, int s) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = s ? a[8 + j] : a[j];
    return pack8(v);
  };
  const bool live = p0 + (r32 >> 4) < npages;
  issue(0, 0);
  for (int t = 0; t < nt; ++t) {
    if (t + 1 < nt) issue(t + 1, (t + 1) & 1);
    if (t + 1 < nt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const bool is_k = t < nk;
    const int wrow = is_k ? perm : r32;
    const char* wt = ring + (t & 1) * TILE;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const bf16x8 w = *reinterpret_cast<const bf16x8*>(wt + wrow * (R * 2) + (((2 * ks + hh) ^ (wrow & 15)) << 4));
      if (is_k) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, ck[ks], acc, 0, 0, 0);
      else acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cv[ks], w, acc, 0, 0, 0);
    }
    __builtin_amdgcn_s_barrier();  // the slot is refilled from the next round on
    if (is_k) {  // acc[8 s + j]: token r32, dim 32 t + 16 s + 8 hh + j
      if (live) {
        bf16_t* o = kt + ((long)(p0 * 16 + r32) * H + h) * D + 32 * t + 8 * hh;
#pragma unroll
        for (int s = 0; s < 2; ++s) *reinterpret_cast<uint4*>(o + 16 * s) = half(acc, s);
      }
    } else {  // acc[8 s + j]: page s, token 8 hh + j, dim 32 (t - nk) + r32
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (p0 + s < npages)
          *reinterpret_cast<uint4*>(vt + (((long)(p0 + s) * H + h) * dv + 32 * (t - nk) + r32) * 16 + 8 * hh) =
              half(acc, s);
    }
  }
  // the shared key part behind the head's own dims
  const int nc = dr / 8;
  for (int i = lane; i < 32 * nc; i += 64) {
    const int tok = i / nc, c = 8 * (i - tok * nc);
    if (p0 + (tok >> 4) < npages)
      *reinterpret_cast<uint4*>(kt + ((long)(p0 * 16 + tok) * H + h) * D + dn + c) =
          *reinterpret_cast<const uint4*>(src(tok) + R + c);
  }
}

// The rotating entries of every head turn in place: rows [T][heads * D], entries rot_off .. rot_off + 2 nf of a head (the
// pairings of rotary_attn.hip).  A token's sines and cosines are evaluated once for all its heads.
template <typename T>
__global__ __launch_bounds__(256) void rotate_heads_kernel(T* __restrict__ x, long stride, int heads, int D,
                                                           const int* __restrict__ positions, const float* __restrict__ freq,
                                                           int nf, int pairs, int rot_off) {
  extern __shared__ float cs[];  // nf cosines, nf sines
  const long t = blockIdx.x;
  const float pos = (float)positions[t];
  for (int i = threadIdx.x; i < nf; i += 256) sincosf(pos * freq[i], cs + nf + i, cs + i);
  __syncthreads();
  for (int e = threadIdx.x; e < heads * nf; e += 256) {
    const int h = e / nf, i = e - h * nf;
    T* p = x + t * stride + (long)h * D + rot_off;
    const int a = pairs ? 2 * i : i, b = pairs ? 2 * i + 1 : i + nf;
    const float u = ldf(p + a), v = ldf(p + b), c = cs[i], s = cs[nf + i];
    stf(p + a, u * c - v * s);
    stf(p + b, v * c + u * s);
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

int k8sllm_hy_latent_expand(void* kt, void* vt, const void* k_cache, int pitch, const int* page_list, int npages, const void* wk,
                            const void* wv, int H, int R, int dn, int dr, int dv, hipStream_t s) {
  if (npages <= 0) return 0;
  if ((R != 128 && R != 256) || dn % 32 || dv % 32 || dn < 32 || dv < 32 || dr % 8 || pitch % 8 || R + dr > pitch || H < 1) return -1;
  const dim3 grid((unsigned)H, (unsigned)((npages + 7) / 8));
  if (R == 128)
    hipLaunchKernelGGL(latent_expand_kernel<128>, grid, dim3(256), 0, s, (bf16_t*)kt, (bf16_t*)vt, (const bf16_t*)k_cache, pitch,
                       page_list, npages, (const bf16_t*)wk, (const bf16_t*)wv, H, dn, dr, dv);
  else
    hipLaunchKernelGGL(latent_expand_kernel<256>, grid, dim3(256), 0, s, (bf16_t*)kt, (bf16_t*)vt, (const bf16_t*)k_cache, pitch,
                       page_list, npages, (const bf16_t*)wk, (const bf16_t*)wv, H, dn, dr, dv);
  return (int)hipGetLastError();
}

int k8sllm_hy_rotate_heads(void* x, long stride, long T, int heads, int D, const int* positions, const float* freq, int nf,
                           int pairs, int rot_off, int f32, hipStream_t s) {
  if (T <= 0 || nf == 0) return 0;
  if (nf < 0 || nf > 4096 || rot_off < 0 || rot_off + 2 * nf > D || heads < 1) return -1;
  const size_t lds = 2 * (size_t)nf * sizeof(float);
  if (f32)
    hipLaunchKernelGGL(rotate_heads_kernel<float>, dim3(T), dim3(256), lds, s, (float*)x, stride, heads, D, positions, freq, nf,
                       pairs, rot_off);
  else
    hipLaunchKernelGGL(rotate_heads_kernel<bf16_t>, dim3(T), dim3(256), lds, s, (bf16_t*)x, stride, heads, D, positions, freq, nf,
                       pairs, rot_off);
  return (int)hipGetLastError();
}
}
