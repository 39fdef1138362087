// Mixture-of-experts plumbing for the Mixtral family:
//   moe_route   softmax over E router logits, top-K, optional renormalisation (one lane per token)
//   moe_align   deterministic counting sort of the T*K (token, slot) pairs by expert, producing
//               expert_offsets[E+1], sorted_idx (position -> flat pair) and inv_idx (pair -> position)
//   gather_rows out[j] = x[idx[j] / div]          (token rows into expert-sorted order)
//   moe_combine out[t] = sum_k w[t][k] * y[inv_idx[t*K + k]]   (fp32 accumulate)
#include "common.h"

namespace k8sllm {

__global__ __launch_bounds__(256) void moe_route_kernel(const float* __restrict__ logits, long T, int E, int K,
                                                        int renorm, int* __restrict__ ids, float* __restrict__ w) {
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  const float* x = logits + t * E;
  float mx = -INFINITY;
  for (int e = 0; e < E; ++e) mx = fmaxf(mx, x[e]);
  float z = 0.f;
  for (int e = 0; e < E; ++e) z += __expf(x[e] - mx);
  uint64_t taken = 0ull;
  float sel = 0.f;
  for (int k = 0; k < K; ++k) {
    int best = -1;
    float bv = -INFINITY;
    for (int e = 0; e < E; ++e)
      if (!((taken >> e) & 1ull) && x[e] > bv) {
        bv = x[e];
        best = e;
      }
    taken |= 1ull << best;
    const float p = __expf(bv - mx) / z;
    ids[t * K + k] = best;
    w[t * K + k] = p;
    sel += p;
  }
  if (renorm)
    for (int k = 0; k < K; ++k) w[t * K + k] /= sel;
}

// MoE decode router in one launch (one workgroup per row): logits = bf16(x . W_router^T) (as the
// library GEMM's bf16 output would be), softmax top-k (+ renormalisation) as moe_route_kernel, and
// the dense per-expert weight row wd[t][e] (0 for an expert the row did not choose) that the grouped
// expert kernels scale their slabs by.  Replaces GEMM + fp32 cast + route + zeros + scatter.
template <int EMAX>
__global__ __launch_bounds__(256) void moe_router_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wr,
                                                         int d, int E, int K, int renorm, int* __restrict__ ids,
                                                         float* __restrict__ w, float* __restrict__ wd) {
  __shared__ float red[4][EMAX];
  const int t = blockIdx.x, tid = threadIdx.x;
  float acc[EMAX];
#pragma unroll
  for (int e = 0; e < EMAX; ++e) acc[e] = 0.f;
  const bf16_t* xr = x + (long)t * d;
  for (int c = tid * 8; c < d; c += 256 * 8) {
    float xv[8];
    unpack8(*reinterpret_cast<const uint4*>(xr + c), xv);
#pragma unroll
    for (int e = 0; e < EMAX; ++e) {
      if (e < E) {
        float wv[8];
        unpack8(*reinterpret_cast<const uint4*>(wr + (long)e * d + c), wv);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[e] = __builtin_fmaf(xv[j], wv[j], acc[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < EMAX; ++e) {
    const float v = wave_sum(acc[e]);
    if ((tid & 63) == 0) red[tid >> 6][e] = v;
  }
  __syncthreads();
  if (tid != 0) return;
  float lg[EMAX];
  float mx = -INFINITY;
  for (int e = 0; e < E; ++e) {
    lg[e] = bf2f(f2bf((red[0][e] + red[1][e]) + (red[2][e] + red[3][e])));
    mx = fmaxf(mx, lg[e]);
  }
  float z = 0.f;
  for (int e = 0; e < E; ++e) z += __expf(lg[e] - mx);
  uint32_t taken = 0u;
  float sel = 0.f, pk[EMAX];
  int bk[EMAX];
  for (int k = 0; k < K; ++k) {
    int best = -1;
    float bv = -INFINITY;
    for (int e = 0; e < E; ++e)
      if (!((taken >> e) & 1u) && lg[e] > bv) {
        bv = lg[e];
        best = e;
      }
    if (best < 0) {  // NaN logits: no comparison holds - take the first untaken expert (a valid id)
      for (best = 0; (taken >> best) & 1u; ++best) {
      }
      bv = lg[best];
    }
    taken |= 1u << best;
    pk[k] = __expf(bv - mx) / z;
    bk[k] = best;
    sel += pk[k];
  }
  for (int e = 0; e < E; ++e) wd[(long)t * E + e] = 0.f;
  for (int k = 0; k < K; ++k) {
    const float p = renorm ? pk[k] / sel : pk[k];
    ids[(long)t * K + k] = bk[k];
    w[(long)t * K + k] = p;
    wd[(long)t * E + bk[k]] = p;
  }
}

constexpr int kAT = 1024;
constexpr int kMaxE = 16;
constexpr int kAlignMaxE = 256;  // up to this many experts with fewer threads (same 64 KiB of counters)

// exclusive scan of one value per thread over an NT-thread workgroup
template <int NT>
__device__ __forceinline__ int block_exscan(int v, int* wsum, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  int pre = 0;
  total = 0;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) {
    const int s = wsum[i];
    if (i < w) pre += s;
    total += s;
  }
  __syncthreads();
  return pre + x - v;
}

// Up to 1024 items and 64 experts (a decode step's), an item per thread: ranks among a wave's items of the same expert come from
// ballots, one lane per expert then sums the waves' counts.  Two barriers where the counters below take two per expert: 128
// items of 8 experts 8.5 -> 2.3 us, 512 of 64 25.8 -> 5.4.
__global__ __launch_bounds__(1024) void moe_align_small_kernel(const int* __restrict__ ids, int n, int E,
                                                               int* __restrict__ offsets, int* __restrict__ sorted_idx,
                                                               int* __restrict__ inv_idx) {
  __shared__ int cnt[16][64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nw = (blockDim.x + 63) >> 6;
  const int e = t < n ? ids[t] : -1;
  int rank = 0, mine = 0;
  for (int i = 0; i < E; ++i) {
    const unsigned long long mask = __ballot(e == i);
    if (e == i) rank = __popcll(mask & ((1ull << lane) - 1));
    if (lane == i) mine = __popcll(mask);
  }
  cnt[wave][lane] = mine;
  __syncthreads();
  if (wave == 0) {
    int tot = 0;
    for (int w = 0; w < nw; ++w) tot += cnt[w][lane];
    int x = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    int at = x - tot;  // lanes past E hold no items
    if (lane < E) offsets[lane] = at;
    if (lane == E - 1) offsets[E] = x;
    for (int w = 0; w < nw; ++w) {
      const int c = cnt[w][lane];
      cnt[w][lane] = at;
      at += c;
    }
  }
  __syncthreads();
  if (t < n) {
    const int pos = cnt[wave][e] + rank;
    sorted_idx[pos] = t;
    inv_idx[t] = pos;
  }
}

// Up to 8 NG experts and kAlignChunkItems items: a workgroup places 1024 of them.  It counts all items and those in front of its own, packed eight bits
// an expert in a thread (hence the limit: at most 63 times four items a thread), sixteen in a wave's sum; ranks among its own come from ballots, as above.  The
// counting is done over by every workgroup, 64 KB of ids at 16384 items, and costs less than one workgroup's placing.  us, one workgroup's counters
// (below) / this: 2000 items of 8 experts 10.1 / 6.9, 16384 19.1 / 7.4, 131072 124 / 17; 16384 of 16 27 / 10.7; 1030 of one 4.9 / 6.1, so from
// three experts on.
constexpr long kAlignChunkItems = 63 * 4096;
template <int NG>
__global__ __launch_bounds__(1024) void moe_align_chunks_kernel(const int* __restrict__ ids, int n, int E, int* __restrict__ offsets,
                                                                int* __restrict__ sorted_idx, int* __restrict__ inv_idx) {
  constexpr int NE = 8 * NG;
  __shared__ int cnt[16][2][NE];  // a wave's items, and those in front of this workgroup's
  __shared__ int own[16][NE];
  __shared__ int start[NE];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, c0 = blockIdx.x * 1024;
  const int e = c0 + t < n ? ids[c0 + t] : -1;
  uint64_t all[NG] = {}, front[NG] = {};
  for (int i = 4 * t; i < n; i += 4096) {
    int v[4];
    if (i + 4 <= n) {
      const int4 q = *reinterpret_cast<const int4*>(ids + i);
      v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = i + k < n ? ids[i + k] : -1;
    }
    uint64_t add[NG] = {};
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int g = 0; g < NG; ++g) add[g] += v[k] >> 3 == g ? 1ull << (8 * (v[k] & 7)) : 0ull;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      all[g] += add[g];
      front[g] += i < c0 ? add[g] : 0ull;
    }
  }
  int rank = 0, mine = 0;
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const unsigned long long mask = __ballot(e == i);
    if (e == i) rank = __popcll(mask & ((1ull << lane) - 1));
    if (lane == i) mine = __popcll(mask);
  }
  if (lane < NE) own[wave][lane] = mine;
  auto sum = [&](const uint64_t (&x)[NG], int* out) {  // over the wave, sixteen bits an expert
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int h = 0; h < 2; ++h) {  // even experts, odd ones
        uint32_t w[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          w[p] = (uint32_t)(x[g] >> (32 * p + 8 * h)) & 0x00ff00ffu;
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) w[p] += __shfl_xor(w[p], o, 64);
          if (lane == 0) {
            out[8 * g + 4 * p + h] = w[p] & 0xffff;
            out[8 * g + 4 * p + h + 2] = w[p] >> 16;
          }
        }
      }
  };
  sum(all, cnt[wave][0]);
  sum(front, cnt[wave][1]);
  __syncthreads();
  if (t < 64) {
    int tot = 0, f = 0;
    if (t < NE)
#pragma unroll
      for (int w = 0; w < 16; ++w) {
        tot += cnt[w][0][t];
        f += cnt[w][1][t];
      }
    int x = tot;
#pragma unroll
    for (int o = 1; o < NE; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (t < NE) start[t] = x - tot + f;
    if (blockIdx.x == 0 && t < E) offsets[t] = x - tot;
    if (blockIdx.x == 0 && t == E - 1) offsets[E] = x;
  }
  __syncthreads();
  if (e >= 0) {
    int pos = start[e] + rank;
#pragma unroll
    for (int w = 0; w < 15; ++w) pos += w < wave ? own[w][e] : 0;
    sorted_idx[pos] = c0 + t;
    inv_idx[c0 + t] = pos;
  }
}

// NT threads x ME experts of per-thread counters fill the 64 KiB of LDS: 1024 x 16 (Mixtral),
// 256 x 64, 64 x 256.
template <int NT, int ME>
__global__ __launch_bounds__(NT) void moe_align_kernel(const int* __restrict__ ids, long n, int E,
                                                       int* __restrict__ offsets, int* __restrict__ sorted_idx,
                                                       int* __restrict__ inv_idx) {
  __shared__ int cnt[ME][NT];
  __shared__ int wsum[NT / 64];
  const int t = threadIdx.x;
  // a thread's items: a multiple of 4, so that ids are read (and inv_idx written) 16 bytes at a time
  const long C = ((n + NT - 1) / NT + 3) & ~3L;
  const long b0 = min(n, t * C), b1 = min(n, b0 + C), b4 = b0 + ((b1 - b0) & ~3L);
  for (int e = 0; e < E; ++e) cnt[e][t] = 0;
#pragma unroll 4
  for (long i = b0; i < b4; i += 4) {
    const int4 e = *reinterpret_cast<const int4*>(ids + i);
    cnt[e.x][t] += 1;
    cnt[e.y][t] += 1;
    cnt[e.z][t] += 1;
    cnt[e.w][t] += 1;
  }
  for (long i = b4; i < b1; ++i) cnt[ids[i]][t] += 1;
  __syncthreads();
  int base = 0;
  for (int e = 0; e < E; ++e) {
    int tot;
    const int ex = block_exscan<NT>(cnt[e][t], wsum, tot);
    if (t == 0) offsets[e] = base;
    cnt[e][t] = base + ex;  // start position of this thread's items of expert e
    base += tot;
  }
  if (t == 0) offsets[E] = base;
#pragma unroll 4
  for (long i = b0; i < b4; i += 4) {
    const int4 e = *reinterpret_cast<const int4*>(ids + i);
    int4 pos;
    pos.x = cnt[e.x][t]++;
    pos.y = cnt[e.y][t]++;
    pos.z = cnt[e.z][t]++;
    pos.w = cnt[e.w][t]++;
    sorted_idx[pos.x] = (int)i;
    sorted_idx[pos.y] = (int)i + 1;
    sorted_idx[pos.z] = (int)i + 2;
    sorted_idx[pos.w] = (int)i + 3;
    *reinterpret_cast<int4*>(inv_idx + i) = pos;
  }
  for (long i = b4; i < b1; ++i) {
    const int pos = cnt[ids[i]][t]++;
    sorted_idx[pos] = (int)i;
    inv_idx[i] = pos;
  }
}

__global__ __launch_bounds__(256) void gather_rows_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
                                                          const int* __restrict__ idx, int d, int div) {
  const long j = blockIdx.x;
  const long src = idx[j] / div;
  const uint4* s = reinterpret_cast<const uint4*>(x + src * d);
  uint4* o = reinterpret_cast<uint4*>(out + j * d);
  for (int i = threadIdx.x; i < (d >> 3); i += 256) o[i] = s[i];
}

__global__ __launch_bounds__(256) void moe_combine_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ y,
                                                          const int* __restrict__ inv_idx,
                                                          const float* __restrict__ w, int K, int d) {
  const long t = blockIdx.x;
  for (int c = threadIdx.x * 8; c < d; c += 256 * 8) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < K; ++k) {
      const float wk = w[t * K + k];
      float v[8];
      unpack8(*reinterpret_cast<const uint4*>(y + (long)inv_idx[t * K + k] * d + c), v);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += wk * v[j];
    }
    *reinterpret_cast<uint4*>(out + t * d + c) = pack8(acc);
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

int k8sllm_moe_route(const void* logits, long T, int E, int K, int renorm, int* topk_ids, float* topk_w,
                     hipStream_t s) {
  if (T <= 0) return 0;
  if (E > 64 || K > E) return -1;
  hipLaunchKernelGGL(moe_route_kernel, dim3((T + 255) / 256), dim3(256), 0, s, (const float*)logits, T, E, K, renorm,
                     topk_ids, topk_w);
  return (int)hipGetLastError();
}

int k8sllm_moe_router(const void* x, const void* wr, long T, int d, int E, int K, int renorm, int* ids, float* w,
                      float* wd, hipStream_t s) {
  if (T <= 0) return 0;
  if (E > 16 || K > E || d % 8 != 0) return -1;
  if (E <= 8)
    hipLaunchKernelGGL(moe_router_kernel<8>, dim3(T), dim3(256), 0, s, (const bf16_t*)x, (const bf16_t*)wr, d, E, K,
                       renorm, ids, w, wd);
  else
    hipLaunchKernelGGL(moe_router_kernel<16>, dim3(T), dim3(256), 0, s, (const bf16_t*)x, (const bf16_t*)wr, d, E, K,
                       renorm, ids, w, wd);
  return (int)hipGetLastError();
}

int k8sllm_moe_align(const int* topk_ids, long n, int E, int* expert_offsets, int* sorted_idx, int* inv_idx,
                     hipStream_t s) {
  if (E > kAlignMaxE) return -1;
  if (n > 0 && n <= 1024 && E <= 64)
    hipLaunchKernelGGL(moe_align_small_kernel, dim3(1), dim3((unsigned)((n + 63) / 64 * 64)), 0, s, topk_ids, (int)n, E, expert_offsets,
                       sorted_idx, inv_idx);
  else if (E >= 3 && E <= 16 && n > 0 && n <= kAlignChunkItems)
    hipLaunchKernelGGL((E <= 8 ? &moe_align_chunks_kernel<1> : &moe_align_chunks_kernel<2>), dim3((unsigned)((n + 1023) / 1024)), dim3(1024), 0,
                       s, topk_ids, (int)n, E, expert_offsets, sorted_idx, inv_idx);
  else if (E <= kMaxE)
    hipLaunchKernelGGL((moe_align_kernel<kAT, kMaxE>), dim3(1), dim3(kAT), 0, s, topk_ids, n, E, expert_offsets,
                       sorted_idx, inv_idx);
  else if (E <= 64)
    hipLaunchKernelGGL((moe_align_kernel<256, 64>), dim3(1), dim3(256), 0, s, topk_ids, n, E, expert_offsets,
                       sorted_idx, inv_idx);
  else
    hipLaunchKernelGGL((moe_align_kernel<64, kAlignMaxE>), dim3(1), dim3(64), 0, s, topk_ids, n, E, expert_offsets,
                       sorted_idx, inv_idx);
  return (int)hipGetLastError();
}

int k8sllm_gather_rows(void* out, const void* x, const int* idx, long n, int d, int div, hipStream_t s) {
  if (n <= 0) return 0;
  if (d % 8 != 0) return -1;
  hipLaunchKernelGGL(gather_rows_kernel, dim3(n), dim3(256), 0, s, (bf16_t*)out, (const bf16_t*)x, idx, d, div);
  return (int)hipGetLastError();
}

int k8sllm_moe_combine(void* out, const void* expert_out, const int* inv_idx, const float* topk_w, long T, int K,
                       int d, hipStream_t s) {
  if (T <= 0) return 0;
  if (d % 8 != 0) return -1;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T), dim3(256), 0, s, (bf16_t*)out, (const bf16_t*)expert_out, inv_idx,
                     topk_w, K, d);
  return (int)hipGetLastError();
}

}  // extern "C"
