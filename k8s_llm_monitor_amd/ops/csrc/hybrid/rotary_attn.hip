// Rotary positions for grouped-query attention over the paged cache of window_attn.hip.
//   rotary_cache   in place on the fused rows [T][Hq*dk | G*dk | G*dv | ...]: the first 2 * nf entries of
//                  every query and key head turn by the angle position * freq[i] (nf frequencies, fp32;
//                  angle, sine and cosine fp32).  pairs == 0: entry i pairs with entry i + nf; pairs == 1:
//                  entry 2i pairs with entry 2i + 1.  Entries from 2 * nf on pass.  q_scale (optional, one
//                  number per query head) multiplies the whole query head in the same pass, before the one
//                  rounding to the activation dtype.  The keys (after the turn) and the values go to the
//                  pages at slots[t] (< 0: not written): keys [blocks][bs][G*dk], values dim-major
//                  [blocks][G][dv][bs].
//   rotary_norm_cache  the same turn with an RMS norm of every query and key head over its dk entries
//                  (fp32, eps inside the root): norm == 1 before the turn, times qw / kw [dk]; norm == 2 after
//                  the turn, no weight; norm == 0 none.  v_from_k: the row has no value columns and the value
//                  pages take the keys as projected (before norm and turn; dv == dk).  One wave per head, the
//                  head staged in LDS as fp32; the token's sines and cosines are evaluated once for all its
//                  heads; the result is rounded to the activation dtype once.  Without rotation, at head
//                  dims 64 / 128 / 256, a lane group per head with wide accesses (head_norm_cache_kernel).
#include <algorithm>

#include "value_pages.h"

namespace k8sllm {

constexpr int kMaxHeadDim = 1024;
constexpr long kTurnRows = 1024;  // from here a workgroup takes up to four rows (7830 rows: 28 us by one, 24.6); fewer would leave CUs idle
constexpr long kFewPairs = 512;  // up to so many turning pairs a row are few (rotary_cache_few_kernel)
// From so many rows of few pairs values go by runs, with the staged form: 269 rows of 4 + 4 heads of 128 4.2 us by rows, 5.2 by runs; 561 of 8 + 8 6.9, 4.8
constexpr long kFewRunRows = 512;
constexpr int kTurns = 512;  // sines and cosines a workgroup of rotary_cache holds at a time

// The norm-only form (norm == 1, nothing turns, head dims of 8 LPH entries): LPH neighbouring lanes hold a head,
// 16 / 32-byte accesses, the mean square by lane adds; a workgroup takes one row.
template <typename T, int LPH>
__global__ __launch_bounds__(256) void head_norm_cache_kernel(T* __restrict__ qkv, long stride, int Hq, int G, int dv,
                                                              const float* __restrict__ qw, const float* __restrict__ kw,
                                                              float eps, const float* __restrict__ q_scale,
                                                              T* __restrict__ k_cache, T* __restrict__ v_cache,
                                                              const int* __restrict__ slots, int bs) {
  constexpr int dk = 8 * LPH;
  const long t = blockIdx.x;
  T* row = qkv + t * stride;
  const int nk = G * dk, nv = G * dv, nh = Hq + G, c = 8 * (threadIdx.x % LPH);
  const long slot = (slots != nullptr && k_cache != nullptr) ? slots[t] : -1;
  for (int h0 = 0; h0 < nh; h0 += 256 / LPH) {  // every lane takes part in the adds; dead heads repeat the last one
    const int h = h0 + threadIdx.x / LPH, hc = min(h, nh - 1);
    T* hd = row + (long)hc * dk + c;
    float x[8], g[8], ss = 0.f;
    load8(hd, x);
    load8((hc >= Hq ? kw : qw) + c, g);
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += x[i] * x[i];
    float inv = 1.0f / sqrtf(lanes_sum<LPH>(ss) / (float)dk + eps);
    if (h >= nh) continue;
    if (h < Hq && q_scale != nullptr) inv *= q_scale[h];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] *= inv * g[i];
    store8(hd, x);
    if (h >= Hq && slot >= 0) store8(k_cache + slot * (long)nk + (long)(h - Hq) * dk + c, x);
  }
  if (slot >= 0)
    for (int i = threadIdx.x; i < nv; i += 256) v_cache[((slot / bs) * nv + i) * bs + slot % bs] = row[(long)nh * dk + i];
}

template <typename T>
__global__ __launch_bounds__(256) void rotary_norm_cache_kernel(T* __restrict__ qkv, long stride, int Hq, int G, int dk,
                                                                int dv, const int* __restrict__ positions,
                                                                const float* __restrict__ freq, int nf, int pairs,
                                                                int norm, const float* __restrict__ qw,
                                                                const float* __restrict__ kw, float eps,
                                                                const float* __restrict__ q_scale,
                                                                T* __restrict__ k_cache, T* __restrict__ v_cache,
                                                                const int* __restrict__ slots, int bs, int v_from_k) {
  extern __shared__ float heads[];  // [4 waves][dk], then the token's nf cosines and nf sines
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  T* row = qkv + t * stride;
  const int nq = Hq * dk, nk = G * dk, nv = G * dv;
  const float pos = (float)positions[t];
  const long slot = (slots != nullptr && k_cache != nullptr) ? slots[t] : -1;
  float* x = heads + wave * dk;
  float* cst = heads + 4 * dk;
  float* snt = cst + nf;
  for (int i = threadIdx.x; i < nf; i += 256) sincosf(pos * freq[i], snt + i, cst + i);  // once for all heads
  __syncthreads();
  // query heads, then key heads (contiguous in the row), a wave per head.  x is this wave's own LDS row: a
  // wave's LDS instructions execute in issue order, so a wave barrier (no reordering by the compiler) is all
  // that lanes reading what other lanes of the wave wrote need.
  for (int h = wave; h < Hq + G; h += 4) {
    T* hd = row + (long)h * dk;
    const bool is_k = h >= Hq;
    const int g = h - Hq;
    float ss = 0.f;
    for (int c = lane; c < dk; c += 64) {
      const float v = ldf(hd + c);
      x[c] = v;
      ss += v * v;
      if (is_k && v_from_k && slot >= 0) v_cache[((slot / bs) * nv + (long)g * dv + c) * bs + slot % bs] = hd[c];
    }
    if (norm == 1) {
      const float inv = 1.0f / sqrtf(wave_sum_dpp(ss) / (float)dk + eps);
      const float* w = is_k ? kw : qw;
      for (int c = lane; c < dk; c += 64) x[c] = x[c] * inv * w[c];
    }
    __builtin_amdgcn_wave_barrier();  // a lane turns pairs whose entries other lanes staged
    for (int i = lane; i < nf; i += 64) {
      const int a = pairs ? 2 * i : i, b = pairs ? 2 * i + 1 : i + nf;
      const float sn = snt[i], cs = cst[i];
      const float u = x[a], v = x[b];
      x[a] = u * cs - v * sn;
      x[b] = v * cs + u * sn;
    }
    __builtin_amdgcn_wave_barrier();
    float mul = 1.f;
    if (norm == 2) {
      float s2 = 0.f;
      for (int c = lane; c < dk; c += 64) s2 += x[c] * x[c];
      mul = 1.0f / sqrtf(wave_sum_dpp(s2) / (float)dk + eps);
    }
    if (!is_k && q_scale != nullptr) mul *= q_scale[h];
    T* kp = (is_k && slot >= 0) ? k_cache + slot * (long)nk + (long)g * dk : nullptr;
    for (int c = lane; c < dk; c += 64) {
      stf(hd + c, x[c] * mul);
      if (kp != nullptr) kp[c] = hd[c];
    }
    __builtin_amdgcn_wave_barrier();  // the next head reuses x
  }
  __syncthreads();  // the value copy below reads nothing the loop wrote, but keeps the workgroup together
  if (!v_from_k && slot >= 0)
    for (int c = threadIdx.x; c < nv; c += 256) v_cache[((slot / bs) * nv + c) * bs + slot % bs] = row[nq + nk + c];
}

// Rows of few turning pairs: a workgroup a row, each pair with sines and cosines of its own, so nothing is staged and no barrier waits.  The same
// products.  us, staged (below) / here: 1 row of 2 + 2 heads of 32 pairs 3.1 / 2.3, of 8 + 4 of 64 2.8 / 3.0; 64 rows of 8 + 2 of 16 3.9 / 3.0; 220 of 2 + 2
// of 16 4.0 / 3.3.
template <typename T>
__global__ __launch_bounds__(256) void rotary_cache_few_kernel(T* __restrict__ qkv, long stride, int Hq, int G, int dk, int dv,
                                                               const int* __restrict__ positions, const float* __restrict__ freq, int nf,
                                                               int pairs, const float* __restrict__ q_scale, T* __restrict__ k_cache,
                                                               T* __restrict__ v_cache, const int* __restrict__ slots, int bs) {
  const long t = blockIdx.x;
  T* row = qkv + t * stride;
  const int nq = Hq * dk, nk = G * dk, nv = G * dv;
  const float pos = (float)positions[t];
  const long slot = (slots != nullptr && k_cache != nullptr) ? slots[t] : -1;
  T* kp = slot >= 0 ? k_cache + slot * (long)nk : nullptr;
  const int rest = dk - 2 * nf;  // entries of a head that do not turn
  for (int e = threadIdx.x; e < (Hq + G) * nf; e += 256) {
    const int h = e / nf, i = e - h * nf;
    const int a = pairs ? 2 * i : i, b = pairs ? 2 * i + 1 : i + nf;
    T* hd = row + (long)h * dk;
    float sn, cs;
    sincosf(pos * freq[i], &sn, &cs);
    const float u = ldf(hd + a), v = ldf(hd + b);
    float x = fmaf(u, cs, -(v * sn)), y = fmaf(v, cs, u * sn);
    if (h < Hq && q_scale != nullptr) {
      x *= q_scale[h];
      y *= q_scale[h];
    }
    stf(hd + a, x);
    stf(hd + b, y);
    if (h >= Hq && kp != nullptr) {
      kp[(h - Hq) * dk + a] = hd[a];
      kp[(h - Hq) * dk + b] = hd[b];
    }
  }
  if (rest > 0) {
    if (q_scale != nullptr)
      for (int e = threadIdx.x; e < Hq * rest; e += 256) {
        const int h = e / rest, c = e - h * rest + 2 * nf;
        T* p = row + (long)h * dk + c;
        stf(p, ldf(p) * q_scale[h]);
      }
    if (kp != nullptr)
      for (int e = threadIdx.x; e < G * rest; e += 256) {
        const int g = e / rest, c = e - g * rest + 2 * nf;
        kp[g * dk + c] = row[nq + g * dk + c];
      }
  }
  if (slot >= 0)
    for (int c = threadIdx.x; c < nv; c += 256) v_cache[((slot / bs) * nv + c) * bs + slot % bs] = row[nq + nk + c];
}

// The sines and cosines of a row's token are evaluated once for all its heads (one for every head and frequency bound the kernel: 20 heads of 64
// frequencies are 1280 of them a row), for the R rows of a workgroup together.  WIDE: eight neighbouring frequencies of a head a thread, 16-byte
// accesses.  The products' roundings are spelled out, so both forms give the same bits.
// Without pages: 7830 rows of 20 heads 28.9 -> 24.6 us, 3749 rows 17.4 -> 15.8, 300 rows of 40 heads 8.2 -> 7.1.
template <typename T, bool WIDE>
__global__ __launch_bounds__(256) void rotary_cache_kernel(T* __restrict__ qkv, long stride, int Hq, int G, int dk,
                                                           int dv, const int* __restrict__ positions,
                                                           const float* __restrict__ freq, int nf, int pairs,
                                                           const float* __restrict__ q_scale,
                                                           T* __restrict__ k_cache, T* __restrict__ v_cache,
                                                           const int* __restrict__ slots, int bs, long rows, int R, int runs) {
  __shared__ alignas(16) float cost[kTurns], sint[kTurns];
  const int nq = Hq * dk, nk = G * dk, nv = G * dv;
  if constexpr (sizeof(T) == 2) {
    if (blockIdx.x < runs) {  // the first workgroups write the values
      write_value_runs(qkv + nq + nk, stride, rows, blockIdx.x, nv, v_cache, slots);
      return;
    }
  }
  const long t0 = (long)(blockIdx.x - runs) * R;
  const int nr = (int)min((long)R, rows - t0);
  const bool cached = slots != nullptr && k_cache != nullptr;
  const int rest = dk - 2 * nf, F = R > 1 ? nf : kTurns;  // rest: entries of a head that do not turn; F: frequencies at a time
  for (int f0 = 0; f0 < nf; f0 += F) {
    const int n = min(nf - f0, F);
    if (f0 > 0) __syncthreads();
    for (int i = threadIdx.x; i < nr * n; i += 256) {
      const int r = i / n;
      sincosf((float)positions[t0 + r] * freq[f0 + i - r * n], sint + i, cost + i);
    }
    __syncthreads();
    // the turning pairs of all query heads, then of all key heads (contiguous in the row): (row, head, i) owns entries (a, b)
    if constexpr (WIDE) {
      const int per = n / 8, one = (Hq + G) * per;
      for (int e = threadIdx.x; e < nr * one; e += 256) {
        const int r = e / one, h = (e - r * one) / per, i = 8 * (e - r * one - h * per);
        const int a = pairs ? 2 * (f0 + i) : f0 + i, b = pairs ? a + 8 : a + nf;
        T* hd = qkv + (t0 + r) * stride + (long)h * dk;
        const float mul = h < Hq && q_scale != nullptr ? q_scale[h] : 1.f;
        float x[8], y[8], cs[8], sn[8];
        load8(hd + a, x);
        load8(hd + b, y);
        load8(cost + r * n + i, cs);
        load8(sint + r * n + i, sn);
        if (pairs) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            float* p = (j < 4 ? x : y) + 2 * (j % 4);
            const float u = p[0], v = p[1];
            p[0] = mul * fmaf(u, cs[j], -(v * sn[j]));
            p[1] = mul * fmaf(v, cs[j], u * sn[j]);
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float u = x[j], v = y[j];
            x[j] = mul * fmaf(u, cs[j], -(v * sn[j]));
            y[j] = mul * fmaf(v, cs[j], u * sn[j]);
          }
        }
        store8(hd + a, x);
        store8(hd + b, y);
        const long slot = h >= Hq && cached ? slots[t0 + r] : -1;
        if (slot >= 0) {
          T* kp = k_cache + slot * nk + (h - Hq) * dk;
          store8(kp + a, x);
          store8(kp + b, y);
        }
      }
    } else {
      T* row = qkv + t0 * stride;
      const long slot = cached ? slots[t0] : -1;
      for (int e = threadIdx.x; e < (Hq + G) * n; e += 256) {
        const int h = e / n, i = e - h * n;
        const int a = pairs ? 2 * (f0 + i) : f0 + i, b = pairs ? a + 1 : a + nf;
        T* hd = row + (long)h * dk;
        const float cs = cost[i], sn = sint[i];
        const float u = ldf(hd + a), v = ldf(hd + b);
        float x = fmaf(u, cs, -(v * sn)), y = fmaf(v, cs, u * sn);
        if (h < Hq && q_scale != nullptr) {
          x *= q_scale[h];
          y *= q_scale[h];
        }
        stf(hd + a, x);
        stf(hd + b, y);
        if (h >= Hq && slot >= 0) {
          T* kp = k_cache + slot * nk + (h - Hq) * dk;
          kp[a] = hd[a];
          kp[b] = hd[b];
        }
      }
    }
  }
  for (int r = 0; r < nr; ++r) {
    T* row = qkv + (t0 + r) * stride;
    const long slot = cached ? slots[t0 + r] : -1;
    if (rest > 0) {
      if (q_scale != nullptr)
        for (int e = threadIdx.x; e < Hq * rest; e += 256) {
          const int h = e / rest, c = e - h * rest + 2 * nf;
          T* p = row + (long)h * dk + c;
          stf(p, ldf(p) * q_scale[h]);
        }
      if (slot >= 0)
        for (int e = threadIdx.x; e < G * rest; e += 256) {
          const int g = e / rest, c = e - g * rest + 2 * nf;
          k_cache[slot * nk + g * dk + c] = row[nq + g * dk + c];
        }
    }
    if (slot >= 0 && !runs)
      for (int c = threadIdx.x; c < nv; c += 256) v_cache[((slot / bs) * nv + c) * bs + slot % bs] = row[nq + nk + c];
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

int k8sllm_hy_rotary_cache(void* qkv, long stride, long T, int Hq, int G, int dk, int dv, const int* positions,
                           const float* freq, int nf, int pairs, const float* q_scale,
                           void* k_cache, void* v_cache, const int* slots, int bs, int singles, int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (nf < 0 || 2 * nf > dk || Hq < 1 || G < 1) return -1;
  const bool few = (long)(Hq + G) * nf <= kFewPairs;
  const int runs = !singles && !f32 && k_cache != nullptr && (!few || T >= kFewRunRows) && value_runs_ok(qkv, stride, (Hq + G) * dk, G * dv, v_cache, slots, T, bs)
                       ? value_groups(T, G * dv)
                       : 0;
  // (fp32 rows with pages, from kTurnRows on, too: 3397 rows of 40 heads of 128 60 us, by four rows a workgroup 74)
  if (runs == 0 && (few || (f32 && T >= kTurnRows && k_cache != nullptr))) {
    if (f32)
      hipLaunchKernelGGL(rotary_cache_few_kernel<float>, dim3((unsigned)T), dim3(256), 0, s, (float*)qkv, stride, Hq, G, dk, dv, positions, freq, nf,
                         pairs, q_scale, (float*)k_cache, (float*)v_cache, slots, bs);
    else
      hipLaunchKernelGGL(rotary_cache_few_kernel<bf16_t>, dim3((unsigned)T), dim3(256), 0, s, (bf16_t*)qkv, stride, Hq, G, dk, dv, positions, freq,
                         nf, pairs, q_scale, (bf16_t*)k_cache, (bf16_t*)v_cache, slots, bs);
    return (int)hipGetLastError();
  }
  const bool wide = nf % 8 == 0 && dk % 8 == 0 && stride % 8 == 0 &&
                    ((reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(k_cache)) & 15) == 0;
  const int R = wide && T >= kTurnRows && nf > 0 && (runs || k_cache == nullptr) ? std::max(1, std::min(4, 256 / nf)) : 1;
  const unsigned grid = (unsigned)((T + R - 1) / R + runs);
#define K8SLLM_TURN(T_, W) \
  hipLaunchKernelGGL((rotary_cache_kernel<T_, W>), dim3(grid), dim3(256), 0, s, (T_*)qkv, stride, Hq, G, dk, dv, positions, \
                     freq, nf, pairs, q_scale, (T_*)k_cache, (T_*)v_cache, slots, bs, T, R, runs)
  if (f32) {
    if (wide) K8SLLM_TURN(float, true);
    else K8SLLM_TURN(float, false);
  } else {
    if (wide) K8SLLM_TURN(bf16_t, true);
    else K8SLLM_TURN(bf16_t, false);
  }
#undef K8SLLM_TURN
  return (int)hipGetLastError();
}

// vec: 8-wide accesses of the rows are aligned (checked by the caller)
int k8sllm_hy_rotary_norm_cache(void* qkv, long stride, long T, int Hq, int G, int dk, int dv, const int* positions,
                                const float* freq, int nf, int pairs, int norm, const float* qw, const float* kw,
                                float eps, const float* q_scale, void* k_cache, void* v_cache, const int* slots, int bs,
                                int v_from_k, int vec, int f32, hipStream_t s) {
  if (T <= 0) return 0;
  if (nf < 0 || 2 * nf > dk || Hq < 1 || G < 1 || dk > kMaxHeadDim || norm < 0 || norm > 2) return -1;
  if (norm == 1 && (qw == nullptr || kw == nullptr)) return -1;
  if (v_from_k && dv != dk) return -1;
  if (nf == 0 && norm == 1 && !v_from_k && vec && (dk == 64 || dk == 128 || dk == 256)) {
#define K8SLLM_HN(T_, LPH)                                                                                            \
  hipLaunchKernelGGL((head_norm_cache_kernel<T_, LPH>), dim3(T), dim3(256), 0, s, (T_*)qkv, stride, Hq, G, dv, qw, kw, eps, \
                     q_scale, (T_*)k_cache, (T_*)v_cache, slots, bs)
    if (f32) {
      if (dk == 64) K8SLLM_HN(float, 8); else if (dk == 128) K8SLLM_HN(float, 16); else K8SLLM_HN(float, 32);
    } else {
      if (dk == 64) K8SLLM_HN(bf16_t, 8); else if (dk == 128) K8SLLM_HN(bf16_t, 16); else K8SLLM_HN(bf16_t, 32);
    }
#undef K8SLLM_HN
    return (int)hipGetLastError();
  }
  const size_t lds = (4 * (size_t)dk + 2 * (size_t)nf) * sizeof(float);
  if (f32)
    hipLaunchKernelGGL(rotary_norm_cache_kernel<float>, dim3(T), dim3(256), lds, s, (float*)qkv, stride, Hq, G, dk, dv,
                       positions, freq, nf, pairs, norm, qw, kw, eps, q_scale, (float*)k_cache, (float*)v_cache, slots, bs,
                       v_from_k);
  else
    hipLaunchKernelGGL(rotary_norm_cache_kernel<bf16_t>, dim3(T), dim3(256), lds, s, (bf16_t*)qkv, stride, Hq, G, dk, dv,
                       positions, freq, nf, pairs, norm, qw, kw, eps, q_scale, (bf16_t*)k_cache, (bf16_t*)v_cache, slots,
                       bs, v_from_k);
  return (int)hipGetLastError();
}
}
