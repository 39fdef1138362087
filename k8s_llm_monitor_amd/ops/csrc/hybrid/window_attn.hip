// Windowed grouped-query attention with a softmax sink over a paged cache (any head size).
//   qk_norm_cache             whole-projection RMSNorm of q and of k in place, k / v -> pages
//   window_attention_prefill  one wave per (chunk row, query head)
//   window_attention_decode   one wave per (sequence, query head)
// Pages: k_cache [blocks][BS][G*dk] (a token's keys contiguous), v_cache [blocks][G][dv][BS] (a value
// dim's BS tokens contiguous: the layout the PV products read along); a sequence's page list is a row of
// block_tables.  Row at position p sees positions max(0, p - window + 1) .. p (window 0: 0 .. p), or with
// ``chunked`` the positions from its chunk's first on: floor(p / window) * window .. p (chunks are counted
// from position 0 of the sequence).  keep > 0 (window form): the first ``keep`` positions of the sequence stay
// visible to every later row besides its window.  cap > 0: a score s (after the scale) becomes cap * tanh(s / cap).
// gate (optional, rows g_stride apart, one logit per query head): a head's output is multiplied by
// sigmoid(gate[row][head]) before its one rounding.  by_value (the bf16 kernels for head sizes of 64 and 128): one logit per value, and the rounded
// output is multiplied by its sigmoid and rounded, as sigmoid_gate does in a pass of its own (7830 rows of 2048 20 us, 3749 12, one row 4).
// The sink is one more softmax term with no value and a fixed score - 0, or a learned unscaled logit
// per query head (sinks[h]): the running maximum starts at that score and the running denominator at 1.  Scores, weights and the output accumulation are fp32.
#include <type_traits>
#include <utility>

#include "stream_rows.h"
#include "value_pages.h"

namespace k8sllm {

constexpr int kMaxVC = 4;  // output dims per lane of the vector decode kernel: dv <= 64 * kMaxVC
constexpr int kMaxDK = 512;
constexpr int kGenVC = 8;  // the any-size kernels: dv <= 64 * kGenVC, dk <= kGenDK
constexpr int kGenDK = 1024;

// tanh from one exponential and one reciprocal: absolute error about 1e-7 (the bf16 kernels' scores; the
// any-size kernels call tanhf)
__device__ __forceinline__ float tanh_exp2(float x) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * 2.88539008177792681f));
}

// NV > 0: up to 256 NV columns of q and of k, kept in registers between the sums and the norms with all loads in flight at once; 0: any
// size, read twice.  The order of the sums is the same.  8192 rows of 2048 + 512 + 512 columns, bf16:
// 44.8 -> 32.2 us, 64 rows 5.8 -> 4.4; 2048 rows of 4096 + 1024 + 1024 25 -> 21.
template <typename T, int NV>
__global__ __launch_bounds__(256) void qk_norm_cache_kernel(T* __restrict__ qkv, long stride,
                                                            const float* __restrict__ qw,
                                                            const float* __restrict__ kw, float eps, int nq, int nk,
                                                            int nv, T* __restrict__ k_cache, T* __restrict__ v_cache,
                                                            const int* __restrict__ slots, int bs, long rows, int runs) {
  __shared__ float red[4];
  if constexpr (sizeof(T) == 2) {
    if (blockIdx.x < runs) {  // the first workgroups write the values
      write_value_runs(qkv + nq + nk, stride, rows, blockIdx.x, nv, v_cache, slots);
      return;
    }
  }
  const long t = blockIdx.x - runs;
  T* row = qkv + t * stride;
  const long slot = (slots != nullptr && k_cache != nullptr) ? slots[t] : -1;
  float sq = 0.f, sk = 0.f;
  if (NV > 0) {
    float q[NV > 0 ? NV : 1], kk[NV > 0 ? NV : 1], wq[NV > 0 ? NV : 1], wk[NV > 0 ? NV : 1];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + 256 * i, cq = min(c, nq - 1), ck = min(c, nk - 1);
      q[i] = ldf(row + cq);
      wq[i] = qw[cq];
      if (256 * i < nk) {
        kk[i] = ldf(row + nq + ck);
        wk[i] = kw[ck];
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + 256 * i;
      if (c < nq) sq += q[i] * q[i];
      if (c < nk) sk += kk[i] * kk[i];
    }
    sq = block_sum<256>(sq, red);
    sk = block_sum<256>(sk, red);
    const float iq = 1.0f / sqrtf(sq / (float)nq + eps), ik = 1.0f / sqrtf(sk / (float)nk + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = threadIdx.x + 256 * i;
      if (c < nq) stf(row + c, q[i] * iq * wq[i]);
      if (c < nk) {
        T kr;
        stf(&kr, kk[i] * ik * wk[i]);
        row[nq + c] = kr;
        if (slot >= 0) k_cache[slot * nk + c] = kr;
      }
    }
  } else {
  for (int c = threadIdx.x; c < nq; c += 256) {
    const float x = ldf(row + c);
    sq += x * x;
  }
  for (int c = threadIdx.x; c < nk; c += 256) {
    const float x = ldf(row + nq + c);
    sk += x * x;
  }
  sq = block_sum<256>(sq, red);
  sk = block_sum<256>(sk, red);
  const float iq = 1.0f / sqrtf(sq / (float)nq + eps), ik = 1.0f / sqrtf(sk / (float)nk + eps);
  for (int c = threadIdx.x; c < nq; c += 256) stf(row + c, ldf(row + c) * iq * qw[c]);
  for (int c = threadIdx.x; c < nk; c += 256) {
    stf(row + nq + c, ldf(row + nq + c) * ik * kw[c]);
    if (slot >= 0) k_cache[slot * nk + c] = row[nq + c];
  }
  }
  if (slot >= 0 && !runs)
    for (int c = threadIdx.x; c < nv; c += 256) v_cache[((slot / bs) * nv + c) * bs + slot % bs] = row[nq + nk + c];
}

// One wave: query q (dk values at q_row) against cached positions [lo, hi) of one kv head.
template <typename T>
__device__ __forceinline__ void attend_wave(T* __restrict__ out_row, const T* __restrict__ q_row,
                                            const T* __restrict__ k_cache, const T* __restrict__ v_cache,
                                            const int* __restrict__ bt, int lo, int hi, int keep, int g, int G,
                                            int dk, int dv, int bs, float scale, float cap, int sink, float sink_z,
                                            float gate, float* q_s, float* p_s) {
  const int lane = threadIdx.x & 63;
  for (int c = lane; c < dk; c += 64) q_s[c] = ldf(q_row + c) * scale;
  __syncthreads();  // one wave per workgroup: orders the LDS writes before the other lanes' reads
  float m = sink ? sink_z : -INFINITY, l = sink ? 1.f : 0.f;  // the sink: one term exp(sink_z - m)
  float acc[kGenVC];
#pragma unroll
  for (int c = 0; c < kGenVC; ++c) acc[c] = 0.f;
  const long krow = (long)G * dk, vrow = (long)G * dv;
  // visible key number i is position i below the kept ones' end, then the window's positions from lo on
  if (keep >= lo) lo = keep = 0;  // nothing lies between them
  const int nvis = keep + hi - lo, skip = lo - keep;
  for (int i0 = 0; i0 < nvis; i0 += 64) {
    const int iv = i0 + lane, j = iv < keep ? iv : iv + skip;
    const bool live = iv < nvis;
    float s = -INFINITY;
    if (live) {
      const T* kp = k_cache + ((long)bt[j / bs] * bs + j % bs) * krow + (long)g * dk;
      float a = 0.f;
      for (int c = 0; c < dk; ++c) a += q_s[c] * ldf(kp + c);
      s = cap > 0.f ? cap * tanhf(a / cap) : a;
    }
    const float mt = fmaxf(m, wave_max_dpp(s));
    const float p = live ? expf(s - mt) : 0.f;
    const float alpha = expf(m - mt);  // m = -inf only before the first key (no sink): exp(-inf) = 0
    l = l * alpha + wave_sum_dpp(p);
    m = mt;
    __syncthreads();  // the previous tile's reads of p_s are done
    p_s[lane] = p;
    __syncthreads();
    const int n = min(64, nvis - i0);
#pragma unroll
    for (int c = 0; c < kGenVC; ++c) {
      const int dcol = lane + 64 * c;
      float a = acc[c] * alpha;
      if (dcol < dv)
        for (int i = 0; i < n; ++i) {
          const int jj = i0 + i < keep ? i0 + i : i0 + i + skip;
          a += p_s[i] * ldf(v_cache + ((long)bt[jj / bs] * vrow + (long)g * dv + dcol) * bs + jj % bs);
        }
      acc[c] = a;
    }
  }
  const float inv = l > 0.f ? gate / l : 0.f;
#pragma unroll
  for (int c = 0; c < kGenVC; ++c) {
    const int dcol = lane + 64 * c;
    if (dcol < dv) stf(out_row + dcol, acc[c] * inv);
  }
}

template <typename T>
__global__ __launch_bounds__(64) void window_prefill_kernel(T* __restrict__ out, const T* __restrict__ qkv,
                                                            long q_stride, const T* __restrict__ k_cache,
                                                            const T* __restrict__ v_cache,
                                                            const int* __restrict__ cu, const int* __restrict__ ctx,
                                                            const int* __restrict__ block_tables, int bt_stride, int S,
                                                            int Hq, int G, int dk, int dv, int bs, float scale,
                                                            int window, int chunked, int keep, float cap, int sink,
                                                            const float* __restrict__ sinks,
                                                            const T* __restrict__ gate, long g_stride) {
  __shared__ float q_s[kGenDK];
  __shared__ float p_s[64];
  const int r = blockIdx.x, h = blockIdx.y;
  const int s = find_segment(cu, S, r);
  const int p = ctx[s] + r - cu[s];
  const int lo = first_key(p, window, chunked);
  attend_wave<T>(out + (long)r * Hq * dv + (long)h * dv, qkv + (long)r * q_stride + (long)h * dk, k_cache, v_cache,
                 block_tables + (long)s * bt_stride, lo, p + 1, keep, h / (Hq / G), G, dk, dv, bs, scale, cap, sink,
                 sinks != nullptr ? sinks[h] : 0.f, gate != nullptr ? sigmoid_f(ldf(gate + (long)r * g_stride + h)) : 1.f,
                 q_s, p_s);
}

template <typename T>
__global__ __launch_bounds__(64) void window_decode_kernel(T* __restrict__ out, const T* __restrict__ qkv,
                                                           long q_stride, const T* __restrict__ k_cache,
                                                           const T* __restrict__ v_cache,
                                                           const int* __restrict__ block_tables, int bt_stride,
                                                           const int* __restrict__ seq_lens, int Hq, int G, int dk,
                                                           int dv, int bs, float scale, int window, int chunked,
                                                           int keep, float cap, int sink,
                                                           const float* __restrict__ sinks,
                                                           const T* __restrict__ gate, long g_stride) {
  __shared__ float q_s[kGenDK];
  __shared__ float p_s[64];
  const int b = blockIdx.x, h = blockIdx.y;
  const int n = seq_lens[b];
  T* o = out + (long)b * Hq * dv + (long)h * dv;
  if (n <= 0) {  // padding row of a decode bucket
    for (int c = threadIdx.x; c < dv; c += 64) stf(o + c, 0.f);
    return;
  }
  const int lo = first_key(n - 1, window, chunked);
  attend_wave<T>(o, qkv + (long)b * q_stride + (long)h * dk, k_cache, v_cache, block_tables + (long)b * bt_stride, lo,
                 n, keep, h / (Hq / G), G, dk, dv, bs, scale, cap, sink, sinks != nullptr ? sinks[h] : 0.f,
                 gate != nullptr ? sigmoid_f(ldf(gate + (long)b * g_stride + h)) : 1.f, q_s, p_s);
}

// bf16 decode with 16-byte loads, 16-token pages: one workgroup (NW = 8 waves; 4 for 8 query heads
// per kv head, whose merge buffers would not fit otherwise) per (sequence, kv head) serves all
// R = Hq / G query heads of that kv head, so every cached key and value is read once.  The waves take
// the window's 64-key tiles (aligned to 64, i.e. four whole pages) in turn and their partial (maximum,
// denominator, output) triples are merged through LDS at the end; only wave 0 starts from the sink's
// (0, 1); scores carry log2 e so that every exponential is one v_exp_f32.  Scores: lane = key, the lane walks its key row in 8-element pieces against the R queries
// held in LDS (fp32).  Values: lane = value dim (+ 64 c); a page's 16 tokens of that dim are two
// 16-byte loads, 2 KiB contiguous per wave; the weights come back from LDS four at a time.
template <int R, int NW>
__global__ __launch_bounds__(64 * NW) void window_decode_vec_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ qkv,
                                                                long q_stride, const bf16_t* __restrict__ k_cache,
                                                                const bf16_t* __restrict__ v_cache,
                                                                const int* __restrict__ block_tables, int bt_stride,
                                                                const int* __restrict__ seq_lens, int Hq, int G, int dk,
                                                                int dv, float scale, int window, int chunked, int keep,
                                                                float cap, int sink, const float* __restrict__ sinks,
                                                                const bf16_t* __restrict__ gate, long g_stride) {
  constexpr int bs = 16;
  __shared__ __attribute__((aligned(16))) float q_s[R * kMaxDK];
  __shared__ __attribute__((aligned(16))) float p_s[NW][R][64];
  __shared__ float ml_s[NW][R][2];
  __shared__ float acc_s[NW][R][64 * kMaxVC];
  const int b = blockIdx.x, g = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = seq_lens[b];
  bf16_t* o = out + (long)b * Hq * dv + (long)g * R * dv;
  if (n <= 0) {  // padding row of a decode bucket
    for (int c = threadIdx.x; c < R * dv; c += 64 * NW) o[c] = 0;
    return;
  }
  const bf16_t* q = qkv + (long)b * q_stride + (long)g * R * dk;
  for (int c = threadIdx.x; c < R * dk; c += 64 * NW) q_s[(c / dk) * kMaxDK + c % dk] = bf2f(q[c]) * (scale * 1.44269504088896341f);  // base-2 scores
  __syncthreads();
  const int* bt = block_tables + (long)b * bt_stride;
  const int lo = first_key(n - 1, window, chunked);
  const float cap2 = cap * 1.44269504088896341f, icap2 = cap > 0.f ? 1.f / cap2 : 0.f;  // base-2 scores
  const bool first = sink && wave == 0;
  float m[R], l[R], acc[R][kMaxVC];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    // the sink's logit is not scaled; scores live in the base-2 domain
    m[r] = first ? (sinks != nullptr ? sinks[g * R + r] * 1.44269504088896341f : 0.f) : -INFINITY;
    l[r] = first ? 1.f : 0.f;
#pragma unroll
    for (int c = 0; c < kMaxVC; ++c) acc[r][c] = 0.f;
  }
  const long krs = (long)G * dk;
  // the tiles that hold kept keys (kt of them, from position 0), then the window's from w0 on
  const int kf = min(keep, n), kt = (kf + 63) >> 6, w0 = max(kt, lo >> 6);
  for (int it = wave;; it += NW) {
    const int j0 = 64 * (it < kt ? it : w0 + it - kt);
    if (j0 >= n) break;
    const int j = j0 + lane;
    const bool valid = (j >= lo || j < keep) && j < n;
    float sc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sc[r] = 0.f;
    if (valid) {
      const bf16_t* kp = k_cache + ((long)bt[j / bs] * bs + j % bs) * krs + (long)g * dk;
      for (int c0 = 0; c0 < dk; c0 += 64) {  // 8 pieces of the key row in flight at a time
        uint4 kq[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (c0 + 8 * u < dk) kq[u] = *reinterpret_cast<const uint4*>(kp + c0 + 8 * u);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int c = c0 + 8 * u;
          if (c < dk) {
            float kv[8];
            unpack8(kq[u], kv);
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const float4 qa = *reinterpret_cast<const float4*>(&q_s[r * kMaxDK + c]);
              const float4 qb = *reinterpret_cast<const float4*>(&q_s[r * kMaxDK + c + 4]);
              sc[r] += kv[0] * qa.x + kv[1] * qa.y + kv[2] * qa.z + kv[3] * qa.w + kv[4] * qb.x + kv[5] * qb.y +
                       kv[6] * qb.z + kv[7] * qb.w;
            }
          }
        }
      }
    }
    // value loads of the tile's pages go out before the softmax arithmetic: 2 x 16 bytes per page and
    // 64 dims (pages at or past the sequence's end are not touched: their weights are zero)
    const int jend = j0 + 64 > lo ? n : kf;  // a tile of kept keys alone: the pages behind them are not needed
    const int npg = min(4, (jend - j0 + bs - 1) / bs);
    uint4 vq[4][kMaxVC][2];
#pragma unroll
    for (int pg = 0; pg < 4; ++pg)
      if (pg < npg) {
        const long base = ((long)bt[j0 / bs + pg] * G + g) * dv;
#pragma unroll
        for (int c = 0; c < kMaxVC; ++c)
          if (lane + 64 * c < dv) {
            const uint4* vp = reinterpret_cast<const uint4*>(v_cache + (base + lane + 64 * c) * bs);
            vq[pg][c][0] = vp[0];
            vq[pg][c][1] = vp[1];
          }
      }
    __builtin_amdgcn_wave_barrier();  // this wave's previous reads of its p_s rows come first
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (cap > 0.f) sc[r] = cap2 * tanh_exp2(sc[r] * icap2);
      const float sv = valid ? sc[r] : -INFINITY;
      const float mt = fmaxf(m[r], wave_max_dpp(sv));  // the tile holds at least one live key, or m is the sink's
      const float pw = (valid && mt != -INFINITY) ? __builtin_amdgcn_exp2f(sv - mt) : 0.f;
      const float alpha = (m[r] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[r] - mt);
      l[r] = l[r] * alpha + wave_sum_dpp(pw);
      m[r] = mt;
      p_s[wave][r][lane] = pw;
#pragma unroll
      for (int c = 0; c < kMaxVC; ++c) acc[r][c] *= alpha;
    }
    __builtin_amdgcn_wave_barrier();  // a wave's LDS instructions execute in issue order
#pragma unroll
    for (int pg = 0; pg < 4; ++pg)
      if (pg < npg) {
#pragma unroll
        for (int c = 0; c < kMaxVC; ++c)
          if (lane + 64 * c < dv) {
            if (j0 + 16 * pg + 16 > n) {  // the last page's unused end (uniform)
              vq[pg][c][0] = tokens_below(vq[pg][c][0], j0 + 16 * pg, n);
              vq[pg][c][1] = tokens_below(vq[pg][c][1], j0 + 16 * pg + 8, n);
            }
            float vv[16];
            unpack8(vq[pg][c][0], vv);
            unpack8(vq[pg][c][1], vv + 8);
#pragma unroll
            for (int r = 0; r < R; ++r) {
              float a = acc[r][c];
#pragma unroll
              for (int t4 = 0; t4 < 4; ++t4) {
                const float4 pq = *reinterpret_cast<const float4*>(&p_s[wave][r][16 * pg + 4 * t4]);
                a += pq.x * vv[4 * t4] + pq.y * vv[4 * t4 + 1] + pq.z * vv[4 * t4 + 2] + pq.w * vv[4 * t4 + 3];
              }
              acc[r][c] = a;
            }
          }
      }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int c = 0; c < kMaxVC; ++c)
      if (lane + 64 * c < dv) acc_s[wave][r][lane + 64 * c] = acc[r][c];
    if (lane == 0) {
      ml_s[wave][r][0] = m[r];
      ml_s[wave][r][1] = l[r];
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < R * dv; c += 64 * NW) {
    const int r = c / dv, dcol = c - r * dv;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, ml_s[w][r][0]);
    float L = 0.f, val = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = ml_s[w][r][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml_s[w][r][0] - M);
      L += ml_s[w][r][1] * f;
      val += acc_s[w][r][dcol] * f;
    }
    const float gt = gate != nullptr ? sigmoid_f(bf2f(gate[(long)b * g_stride + g * R + r])) : 1.f;
    o[c] = f2bf(L > 0.f ? val / L * gt : 0.f);
  }
}

// t = sum of 8 (4) products v[k] x[N + k], x's elements those of this 16-lane row (DPP row_newbcast), for one or two x at a time; the
// second product first, then the first, the third, ..  The s_nop keeps the two wait states between a vector write and a DPP
// read of the same register, whatever stands in front.
template <int N>
__device__ __forceinline__ void row_dot8(float xa, float xb, const float* v, float& ta, float& tb) {
  asm("s_nop 1\n\t"
      "v_mul_f32_dpp %[ta], %[xa], %[v1] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf\n\t"
      "v_mul_f32_dpp %[tb], %[xb], %[v1] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v0] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v0] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v2] row_newbcast:%[n2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v2] row_newbcast:%[n2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v3] row_newbcast:%[n3] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v3] row_newbcast:%[n3] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v4] row_newbcast:%[n4] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v4] row_newbcast:%[n4] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v5] row_newbcast:%[n5] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v5] row_newbcast:%[n5] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v6] row_newbcast:%[n6] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v6] row_newbcast:%[n6] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v7] row_newbcast:%[n7] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v7] row_newbcast:%[n7] row_mask:0xf bank_mask:0xf\n\t"
      : [ta] "=&v"(ta), [tb] "=&v"(tb)
      : [xa] "v"(xa), [xb] "v"(xb), [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [v4] "v"(v[4]), [v5] "v"(v[5]), [v6] "v"(v[6]), [v7] "v"(v[7]), [n0] "n"(N + 0), [n1] "n"(N + 1), [n2] "n"(N + 2), [n3] "n"(N + 3), [n4] "n"(N + 4), [n5] "n"(N + 5), [n6] "n"(N + 6), [n7] "n"(N + 7));
}
template <int N>
__device__ __forceinline__ void row_dot8(float xa, const float* v, float& ta) {
  asm("s_nop 1\n\t"
      "v_mul_f32_dpp %[ta], %[xa], %[v1] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v0] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v2] row_newbcast:%[n2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v3] row_newbcast:%[n3] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v4] row_newbcast:%[n4] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v5] row_newbcast:%[n5] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v6] row_newbcast:%[n6] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v7] row_newbcast:%[n7] row_mask:0xf bank_mask:0xf\n\t"
      : [ta] "=&v"(ta)
      : [xa] "v"(xa), [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [v4] "v"(v[4]), [v5] "v"(v[5]), [v6] "v"(v[6]), [v7] "v"(v[7]), [n0] "n"(N + 0), [n1] "n"(N + 1), [n2] "n"(N + 2), [n3] "n"(N + 3), [n4] "n"(N + 4), [n5] "n"(N + 5), [n6] "n"(N + 6), [n7] "n"(N + 7));
}
template <int N>
__device__ __forceinline__ void row_dot4(float xa, float xb, const float* v, float& ta, float& tb) {
  asm("s_nop 1\n\t"
      "v_mul_f32_dpp %[ta], %[xa], %[v1] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf\n\t"
      "v_mul_f32_dpp %[tb], %[xb], %[v1] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v0] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v0] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v2] row_newbcast:%[n2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v2] row_newbcast:%[n2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v3] row_newbcast:%[n3] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[tb], %[xb], %[v3] row_newbcast:%[n3] row_mask:0xf bank_mask:0xf\n\t"
      : [ta] "=&v"(ta), [tb] "=&v"(tb)
      : [xa] "v"(xa), [xb] "v"(xb), [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [n0] "n"(N + 0), [n1] "n"(N + 1), [n2] "n"(N + 2), [n3] "n"(N + 3));
}
template <int N>
__device__ __forceinline__ void row_dot4(float xa, const float* v, float& ta) {
  asm("s_nop 1\n\t"
      "v_mul_f32_dpp %[ta], %[xa], %[v1] row_newbcast:%[n1] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v0] row_newbcast:%[n0] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v2] row_newbcast:%[n2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %[ta], %[xa], %[v3] row_newbcast:%[n3] row_mask:0xf bank_mask:0xf\n\t"
      : [ta] "=&v"(ta)
      : [xa] "v"(xa), [v0] "v"(v[0]), [v1] "v"(v[1]), [v2] "v"(v[2]), [v3] "v"(v[3]), [n0] "n"(N + 0), [n1] "n"(N + 1), [n2] "n"(N + 2), [n3] "n"(N + 3));
}
template <int N, typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// Query heads that a workgroup of the kernel below takes, R sharing a kv head: the fewest that leave each of 256 compute units at most one
// workgroup, all that its registers and LDS let it run.  A wave's tile costs its instructions for every head, and its keys' loads once for each
// workgroup.  us, all heads / half / one of four: 1 sequence of 333 keys, 8 heads on 2 10.9 / 7.8 / 6.6; 8 of 1500, 16 on 4 30.6 / 22.6 /
// 19.3; 24 of 1500, 16 on 4 35.6 / 27.5 / 36.3; 64 of 1024 35.0 / 39.9 / 58.8; 16 of 1500, 8 heads on one, all / 2 / 1: 58.2 / 28.6 / 25.5.
inline int decode_heads(long B, int Hq, int R) {
  for (int heads : {1, 2})
    if (heads < R && R % heads == 0 && B * Hq <= 256L * heads) return heads;
  return R;
}

// The same for head sizes of 64 and 128, without the LDS reads that bound it (a tile of 64 keys took a wave 256 16-byte reads of
// queries and weights that all lanes share): each 16-lane row holds all dims of the queries, 16 to a register, and a page's 16
// weights in one, and the multiply-adds pick the element by their DPP row broadcast.  Sums in the same order: the same bits.
// A tile's keys come to LDS by whole rows, 16 lanes a row, and the next tile's while this one is multiplied; a lane then reads its own.
// Loads of a row a lane met 64 rows at a time, which is 64 cycles of the load path each, and a page's values, loaded behind a
// branch, waited for the page before.  The same bits.  us over pages from memory, keys by a row a lane and all heads a workgroup / now at
// decode_heads' choice, heads of 128: 1 sequence of 333 keys, 8 heads on 2 13.7 / 6.6; of 4000, 16 on 4 84 / 36; 24 of 1500 45 / 28; 64 of 1000
// 39 / 34 (3.9 TB/s); 256 of 300 66 / 52; 64 of 1000, 16 heads on 2 55 / 45.
// (In a step of 64 sequences behind 2048 tokens, window 1024, 46.8 / 44.3 a layer: 17 tiles of keys are three rounds of eight waves.)
// A page's address is the wave's own, in scalar registers, and a lane adds one of a few offsets: an address a lane took up to 44 vector registers.
// PER_CU: heads of 64, four a workgroup, in 128 registers (4 of 165 spilled), so that two share a compute unit once there is more than
// one for each.  us, before the keys came through LDS / 165 registers / this, 32 heads on 8: 256 sequences of 64 keys 31 / 36 / 25, of 300 50 / 56 /
// 44, of 1000 118 / 117 / 116; 16 on 4, 64 of 1000, one workgroup each, 23.0 / 18.9 / 20.0.
template <int R, int NW, int DKC, int VC, int PER_CU = 1>
__global__ __launch_bounds__(64 * NW, PER_CU * NW / 4) void window_decode_row_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ qkv,
                                                                long q_stride, const bf16_t* __restrict__ k_cache,
                                                                const bf16_t* __restrict__ v_cache,
                                                                const int* __restrict__ block_tables, int bt_stride,
                                                                const int* __restrict__ seq_lens, int Hq, int G, float scale, int window, int chunked, int keep,
                                                                float cap, int sink, const float* __restrict__ sinks,
                                                                const bf16_t* __restrict__ gate, long g_stride, int by_value) {
  constexpr int bs = 16;
  __shared__ float ml_s[NW][R][2];
  constexpr int dk = 64 * DKC, dv = 64 * VC;
  static_assert(4 * R * dv <= 128 * dk, "");
  __shared__ __attribute__((aligned(1024))) char k_s[NW][128 * dk];  // a wave's tile of keys; its results when the keys are done
  const int b = blockIdx.x, h0 = blockIdx.y * R, g = h0 / (Hq / G), lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = seq_lens[b];
  bf16_t* o = out + (long)b * Hq * dv + (long)h0 * dv;
  if (n <= 0) {  // padding row of a decode bucket
    for (int c = threadIdx.x; c < R * dv; c += 64 * NW) o[c] = 0;
    return;
  }
  const int* bt = block_tables + (long)b * bt_stride;
  const int lo = first_key(n - 1, window, chunked);
  const long krs = (long)G * dk;
  // the tiles that hold kept keys (kt of them, from position 0), then the window's from w0 on
  const int kf = min(keep, n), kt = (kf + 63) >> 6, w0 = max(kt, lo >> 6);
  auto tile = [&](int it) { return 64 * (it < kt ? it : w0 + it - kt); };
  // keys j0 .. j0 + 63 to LDS, a row's 16-byte chunks turned by the row; pages without a key to be seen: the newest one's instead.
  // A page's address is the wave's, a lane adds one of PER offsets.
  constexpr int LPK = dk / 8, RPI = 64 / LPK, PER = bs / RPI;
  auto turn = [](int r) { return DKC == 2 ? r & 15 : (r >> 1) & 7; };
  uint32_t koff[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) koff[i] = 2 * (uint32_t)((i * RPI + lane / LPK) * (int)krs + 8 * ((lane % LPK) ^ turn(i * RPI + lane / LPK)));
  auto stage = [&](int j0) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int f = j0 + 16 * p;
      const long page = (long)bt[((f < n) & ((f + 15 >= lo) | (f < keep)) ? f : n - 1) / bs] * bs;
      const char* base = reinterpret_cast<const char*>(k_cache + page * krs + (long)g * dk);
#pragma unroll
      for (int i = 0; i < PER; ++i) load_piece(k_s[wave] + 1024 * (PER * p + i), reinterpret_cast<const bf16_t*>(base + koff[i]));
    }
  };
  int it = wave, j0 = tile(it);
  if (j0 < n) stage(j0);
  // loads from an argument may sink past a barrier into the branch of their use: an address of unknown origin
  uint32_t vlo = (uint32_t)reinterpret_cast<uint64_t>(v_cache), vhi = (uint32_t)(reinterpret_cast<uint64_t>(v_cache) >> 32);
  asm volatile("" : "+v"(vlo), "+v"(vhi));
  const long values = (long)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(vhi) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane(vlo));
  const bf16_t* q = qkv + (long)b * q_stride + (long)h0 * dk;
  // base-2 scores; lane l of every 16-lane row holds the queries' dims 16 i + l % 16
  float qr[R][4 * DKC];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int i = 0; i < 4 * DKC; ++i) qr[r][i] = bf2f(q[r * dk + 16 * i + (lane & 15)]) * (scale * 1.44269504088896341f);
  const float cap2 = cap * 1.44269504088896341f, icap2 = cap > 0.f ? 1.f / cap2 : 0.f;  // base-2 scores
  const bool first = sink && wave == 0;
  float m[R], l[R], acc[R][VC];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    // the sink's logit is not scaled; scores live in the base-2 domain
    m[r] = first ? (sinks != nullptr ? sinks[h0 + r] * 1.44269504088896341f : 0.f) : -INFINITY;
    l[r] = first ? 1.f : 0.f;
#pragma unroll
    for (int c = 0; c < VC; ++c) acc[r][c] = 0.f;
  }
  auto step = [&](int next, auto more) {  // no load behind a branch: the tile's values, then the next tile's keys, are on their way meanwhile
    const int j = j0 + lane;
    const bool valid = (j >= lo || j < keep) && j < n;
    float sc[R], p[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sc[r] = 0.f;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tile's keys are there
    // value loads of the tile's pages go out before the arithmetic: 2 x 16 bytes per page and
    // 64 dims (pages at or past the sequence's end are not touched: the last one is read again, and nothing multiplies it)
    const int jend = j0 + 64 > lo ? n : kf;  // a tile of kept keys alone: the pages behind them are not needed
    const int npg = min(4, (jend - j0 + bs - 1) / bs);
    uint4 vq[4][VC][2], kr[8 * DKC];
#pragma unroll
    for (int pg = 0; pg < 4; ++pg) {
      const long base = values + 2 * bs * (((long)bt[j0 / bs + min(pg, npg - 1)] * G + g) * dv);
#pragma unroll
      for (int c = 0; c < VC; ++c) {
        using Raw = unsigned __attribute__((ext_vector_type(4)));
        const auto vp = reinterpret_cast<__attribute__((address_space(1))) const Raw*>(base + 2 * bs * 64 * c + (long)(2 * bs * (uint32_t)lane));
        vq[pg][c][0] = __builtin_bit_cast(uint4, Raw(vp[0]));
        vq[pg][c][1] = __builtin_bit_cast(uint4, Raw(vp[1]));
      }
    }
#pragma unroll
    for (int u = 0; u < 8 * DKC; ++u) kr[u] = *reinterpret_cast<const uint4*>(k_s[wave] + 2 * dk * lane + 16 * (u ^ turn(lane)));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the keys have been read
    if constexpr (decltype(more)::value) stage(next);
    static_for<8 * DKC>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      float kv[8];
      unpack8(kr[u], kv);
      constexpr int h = 8 * (u & 1);
      if constexpr (R == 1) {
        float t;
        row_dot8<h>(qr[0][u / 2], kv, t);
        sc[0] += t;
      } else {
#pragma unroll
        for (int r = 0; r < R; r += 2) {
          float t0, t1;
          row_dot8<h>(qr[r][u / 2], qr[r + 1][u / 2], kv, t0, t1);
          sc[r] += t0;
          sc[r + 1] += t1;
        }
      }
    });
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (cap > 0.f) sc[r] = cap2 * tanh_exp2(sc[r] * icap2);
      const float sv = valid ? sc[r] : -INFINITY;
      const float mt = fmaxf(m[r], wave_max_dpp(sv));  // the tile holds at least one live key, or m is the sink's
      const float pw = (valid && mt != -INFINITY) ? __builtin_amdgcn_exp2f(sv - mt) : 0.f;
      const float alpha = (m[r] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m[r] - mt);
      l[r] = l[r] * alpha + wave_sum_dpp(pw);
      m[r] = mt;
      p[r] = pw;
#pragma unroll
      for (int c = 0; c < VC; ++c) acc[r][c] *= alpha;
    }
#pragma unroll
    for (int pg = 0; pg < 4; ++pg)
      if (pg < npg) {
        float pr[R];  // every row of lanes: the page's 16 weights
#pragma unroll
        for (int r = 0; r < R; ++r) pr[r] = __shfl(p[r], 16 * pg + (lane & 15), kWave);
#pragma unroll
        for (int c = 0; c < VC; ++c) {
          if (j0 + 16 * pg + 16 > n) {  // the last page's unused end (uniform)
            vq[pg][c][0] = tokens_below(vq[pg][c][0], j0 + 16 * pg, n);
            vq[pg][c][1] = tokens_below(vq[pg][c][1], j0 + 16 * pg + 8, n);
          }
          float vv[16];
          unpack8(vq[pg][c][0], vv);
          unpack8(vq[pg][c][1], vv + 8);
          static_for<4>([&](auto tc) {
            constexpr int t4 = 4 * decltype(tc)::value;
            if constexpr (R == 1) {
              float t;
              row_dot4<t4>(pr[0], vv + t4, t);
              acc[0][c] += t;
            } else {
#pragma unroll
              for (int r = 0; r < R; r += 2) {
                float t0, t1;
                row_dot4<t4>(pr[r], pr[r + 1], vv + t4, t0, t1);
                acc[r][c] += t0;
                acc[r + 1][c] += t1;
              }
            }
          });
        }
      }
  };
  if (j0 < n) {
    for (int next; (next = tile(it + NW)) < n; it += NW, j0 = next) step(next, std::true_type{});
    step(0, std::false_type{});
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int c = 0; c < VC; ++c)
      reinterpret_cast<float*>(k_s[wave])[r * dv + lane + 64 * c] = acc[r][c];
    if (lane == 0) {
      ml_s[wave][r][0] = m[r];
      ml_s[wave][r][1] = l[r];
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < R * dv; c += 64 * NW) {
    const int r = c / dv, dcol = c - r * dv;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, ml_s[w][r][0]);
    float L = 0.f, val = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = ml_s[w][r][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml_s[w][r][0] - M);
      L += ml_s[w][r][1] * f;
      val += reinterpret_cast<const float*>(k_s[w])[r * dv + dcol] * f;
    }
    const float gt = gate != nullptr && !by_value ? sigmoid_f(bf2f(gate[(long)b * g_stride + h0 + r])) : 1.f;
    const bf16_t x = f2bf(L > 0.f ? val / L * gt : 0.f);
    o[c] = by_value ? f2bf(bf2f(x) * sigmoid_f(bf2f(gate[(long)b * g_stride + (long)h0 * dv + c]))) : x;
  }
}

// bf16 prefill on the matrix cores, head sizes that are multiples of 32 (keys) / 16 (values).
// One wave = 16 consecutive chunk rows of one sequence x one query head; key tiles of 16.
//   S^T[key][q]  = K Q^T      v_mfma_f32_16x16x32_bf16: A = K rows (16-byte loads straight from the
//                             pages), B = the wave's Q rows (held in registers for the whole loop)
//   O^T[d][q]   += V^T P^T    v_mfma_f32_16x16x16_bf16: B = the score accumulator itself (query on
//                             the lane, 4 keys per lane: the C layout of S^T IS the B layout of P^T),
//                             A = V^T, 8-byte loads from the d-major V page (tokens contiguous)
// With the query on the lane the running maximum, denominator and the rescale of O are lane-local
// (two xor-shuffles per reduction).  Scores, weights and sums are fp32 (base-2 exponentials: the
// scale carries log2 e); P is rounded to bf16 for the PV product.
// CAP 1: capped scores.  CAP 2: capped scores with a cap up to kMaxCapPlain and no sink: a score lies within
// +-cap, so exp(score) cannot leave the fp32 (or bf16) range and the softmax is taken as it stands, without a
// running maximum, rescaling or a cross-lane sum per tile (the lanes' parts of the denominator meet at the
// end); only tiles at a row's first or last key are masked.
constexpr float kMaxCapPlain = 60.f;
// The LDS-staged kernel of window_flash.hip takes a step that has enough (row, head) pairs to fill the chip with its
// 256 pairs per workgroup, or rows that may see enough keys for the shared tiles to pay with few workgroups.  Register
// kernel at its better width -> staged kernel, us (128-wide heads): 13 prompts x 120, 8 heads (12480 pairs, 120 keys)
// 9.5 -> 13.4; x 250 22.4 -> 17.7; x 500 52 -> 26; one prompt of 512, 8 heads 20.9 -> 22.2; 1024 39 -> 35; 64 rows
// behind 2000 keys, 16 heads 72 -> 64.  mfma = kFlashForced asks for it at any size (tests, measurements), 2 for the
// register kernel whatever the size.
constexpr long kFlashPairs = 16 * 1024;
constexpr long kFlashKeys = 1024;
constexpr int kFlashForced = 256;
// WH = 4: four waves, each with its own query head of one kv head, share that head's keys and values.  Register loads of K
// in fragment order touch 16 rows per 16 lanes, which the load path takes at about a quarter of its rate, and every head
// fetched every key for itself: 4 x 2048 rows, 16 heads over 4, window 1024: 218 us; through LDS 154.  4 x 1024, 32 heads over
// 8: 164 -> 122.  The products and their order are the same, so are the bits.  Smaller steps keep one wave per workgroup:
// there a wave's chain bounds, and the barriers lengthen it (3 x 64 rows: 9.9 us, shared 12.6).
template <int DK, int DV, int QT, int CAP, int WH>
__global__ __launch_bounds__(WH ? 64 * WH : 64, WH == 0 || QT == 4 ? 1 : 3) void window_prefill_mfma_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ qkv, long q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int* __restrict__ cu, const int* __restrict__ ctx,
    const int* __restrict__ block_tables, int bt_stride, int S, int Hq, int G, float scale, int window,
    int chunked, int keep, float cap, int sink, const float* __restrict__ sinks, const bf16_t* __restrict__ gate,
    long g_stride, int by_value) {
  // pages hold 16 tokens; scores live in the base-2 domain (scale * log2 e folded in) so that every
  // exponential is one v_exp_f32
  const float sc2 = scale * 1.44269504088896341f;
  const float cap2 = CAP ? cap * 1.44269504088896341f : 0.f, icap = CAP ? scale / cap : 0.f;
  constexpr int QB = 16 * QT;  // query rows per wave: QT tiles of 16 share every K and V^T fragment
  int tile = blockIdx.x, s = 0, n = 0;
  for (; s < S; ++s) {  // q-blocks are numbered segment by segment
    n = cu[s + 1] - cu[s];
    const int nt = (n + QB - 1) / QB;
    if (tile < nt) break;
    tile -= nt;
  }
  if (s >= S) return;
  const int q0 = tile * QB, nq = min(QB, n - q0);
  constexpr bool SHARED = WH > 0;
  const int wave = SHARED ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int h = SHARED ? blockIdx.y * WH + wave : blockIdx.y, g = h / (Hq / G);
  const int lane = threadIdx.x & 63, c16 = lane & 15, quad = lane >> 4;
  const int* bt = block_tables + (long)s * bt_stride;
  const int row0 = cu[s] + q0, p0 = ctx[s] + q0;
  int my_p[QT], my_lo[QT];
  bool q_live[QT];
  bf16x8 qf[QT][DK / 32];
  f32x4 oacc[QT][DV / 16];
  float m[QT], l[QT];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int myq = min(16 * t + c16, nq - 1);
    my_p[t] = p0 + myq;
    my_lo[t] = first_key(my_p[t], window, chunked);
    q_live[t] = 16 * t + c16 < nq;
    const bf16_t* qrow = qkv + (long)(row0 + myq) * q_stride + (long)h * DK;
#pragma unroll
    for (int ks = 0; ks < DK / 32; ++ks) qf[t][ks] = *reinterpret_cast<const bf16x8*>(qrow + 32 * ks + 8 * quad);
#pragma unroll
    for (int dt = 0; dt < DV / 16; ++dt) oacc[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[t] = sink ? (sinks != nullptr ? sinks[h] * 1.44269504088896341f : 0.f) : -INFINITY;
    l[t] = sink ? 1.f : 0.f;
  }
  const int lo_max = first_key(p0 + nq - 1, window, chunked);  // from here to p0: keys that every row of the tile sees
  const float k1 = CAP ? icap * 2.88539008177792681f : 0.f;
  const int lo_t = first_key(p0, window, chunked), hi = p0 + nq;
  const long krs = (long)G * DK, vrs = (long)G * DV;
  // key tiles: those that hold kept keys (up to kend), then the window's from wfirst on
  const int kend = (min(keep, hi) + 15) & ~15, wfirst = max(kend, lo_t & ~15);
  const int jfirst = kend > 0 ? 0 : wfirst;
  auto next_tile = [&](int j) {
    j += 16;
    return j >= kend && j < wfirst ? wfirst : j;
  };
  // SHARED: two tiles at a time come to LDS for all waves (stream_rows.h: K in pieces of 16 keys x 32 dims, V^T as the page has it), a
  // ring of three such stages with one barrier each; two are on their way while one is computed, the next one's page ids behind them.
  // Else registers: while a tile is computed, the K and V^T fragments of the next are in flight, and the page id of the one after it.
  constexpr int KP = DK / 32, VP = DV / 32, W = SHARED ? WH : 1, PK = 2 * KP / W, PV = 2 * VP / W, STAGE = 2 * (KP + VP) * 1024;
  __shared__ __attribute__((aligned(1024))) char ring[SHARED ? 3 * STAGE : 16];
  const bf16_t* kbase = k_cache + (long)g * DK + (SHARED ? piece_k() : 8 * quad);
  const bf16_t* vbase = v_cache + (long)g * DV * 16 + (SHARED ? 8 * lane : 16 * c16 + 4 * quad);
  constexpr int AHEAD = SHARED ? 2 : 1;
  int ji = jfirst, jn[AHEAD], pg[AHEAD];  // the tiles that are loaded next and their pages
  auto pages = [&]() {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      jn[u] = ji;
      pg[u] = bt[min(ji, hi - 1) >> 4];
      ji = next_tile(ji);
    }
  };
  bf16x8 kn[DK / 32];
  s16x4 vn[DV / 16];
  auto issue = [&](int slot) {  // (a tile past the last key: the last page once more)
    if constexpr (SHARED) {
      char* dst = ring + slot * STAGE;
#pragma unroll
      for (int q = 0; q < PK; ++q) {
        const int i = wave + W * q, u = i / KP, ks = i % KP;
        const int j = u ? jn[AHEAD - 1] : jn[0];
        const long row = ((long)(u ? pg[AHEAD - 1] : pg[0]) << 4) + (min(j + piece_row(), hi - 1) & 15);
        load_piece(dst + i * 1024, kbase + row * krs + 32 * ks);
      }
#pragma unroll
      for (int q = 0; q < PV; ++q) {
        const int i = wave + W * q, u = i / VP, dp = i % VP;
        load_piece(dst + (2 * KP + i) * 1024, vbase + (long)(u ? pg[AHEAD - 1] : pg[0]) * vrs * 16 + 512 * dp);
      }
    } else {
      const bf16_t* krow = kbase + (((long)pg[0] << 4) + (min(jn[0] + c16, hi - 1) & 15)) * krs;
#pragma unroll
      for (int ks = 0; ks < DK / 32; ++ks) kn[ks] = *reinterpret_cast<const bf16x8*>(krow + 32 * ks);
      const bf16_t* vpg = vbase + (long)pg[0] * vrs * 16;
#pragma unroll
      for (int dt = 0; dt < DV / 16; ++dt) vn[dt] = *reinterpret_cast<const s16x4*>(vpg + dt * 256);
    }
  };
  const int kfrag = piece_frag(), vfrag = c16 * 32 + quad * 8;
  pages();
  issue(0);
  pages();
  if (SHARED) {
    issue(1);
    pages();
  }
  int slot = 0;
  for (int j2 = jfirst; j2 < hi;) {
   const char* src = ring;
   if (SHARED) {
    loads_left<PK + PV>();  // this stage's, of this wave
    __builtin_amdgcn_s_barrier();  // of all waves; and the slot filled next has been read
    issue(slot == 0 ? 2 : slot - 1);
    pages();
    src = ring + slot * STAGE;
    slot = slot == 2 ? 0 : slot + 1;
   }
#pragma unroll 1
   for (int u = 0; u < AHEAD; ++u) {
    const int j0 = j2;
    j2 = next_tile(j2);
    if (j0 >= hi) break;
    bf16x8 kf[DK / 32];
    s16x4 vf[DV / 16];
#pragma unroll
    for (int ks = 0; ks < DK / 32; ++ks) kf[ks] = SHARED ? *reinterpret_cast<const bf16x8*>(src + (u * KP + ks) * 1024 + kfrag) : kn[ks];
    if constexpr (!SHARED) {
#pragma unroll
      for (int dt = 0; dt < DV / 16; ++dt) vf[dt] = vn[dt];
      if (j2 < hi) {
        issue(0);
        pages();
      }
    }
    f32x4 scores[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) scores[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < DK / 32; ++ks)
#pragma unroll
      for (int t = 0; t < QT; ++t) scores[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks], qf[t][ks], scores[t], 0, 0, 0);
    if constexpr (SHARED) {  // (behind the scores' products, which need the keys only)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int dt = 0; dt < DV / 16; ++dt) vf[dt] = *reinterpret_cast<const s16x4*>(src + (2 * KP + u * VP) * 1024 + dt * 512 + vfrag);
    }
    if (j0 + 16 > hi) {  // the last page's unused end (wave-uniform)
      const int j = j0 + 4 * quad;
      const uint32_t ma = pair_below(j, hi), mb = pair_below(j + 2, hi);
#pragma unroll
      for (int dt = 0; dt < DV / 16; ++dt) {
        const uint2 v = __builtin_bit_cast(uint2, vf[dt]);
        vf[dt] = __builtin_bit_cast(s16x4, make_uint2(v.x & ma, v.y & mb));
      }
    }
    s16x4 pb[QT];
    float alpha[QT];
    bool rescale[QT];
    const bool inner = (j0 >= lo_max || j0 + 15 < keep) && j0 + 15 <= p0;  // wave-uniform: every row sees every key
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const f32x4 sacc = scores[t];
      if constexpr (CAP == 2) {
        float pv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)  // exp(cap tanh(s / cap)) in base 2
          pv[i] = __builtin_amdgcn_exp2f(cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(sacc[i] * k1)));
        if (!inner) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int j = j0 + 4 * quad + i;
            if ((j < my_lo[t] && j >= keep) || j > my_p[t]) pv[i] = 0.f;
          }
        }
        l[t] += (pv[0] + pv[1]) + (pv[2] + pv[3]);
#pragma unroll
        for (int i = 0; i < 4; ++i) pb[t][i] = (short)f2bf(pv[i]);
        continue;
      }
      float sv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) sv[i] = CAP ? cap2 * tanh_exp2(sacc[i] * icap) : sacc[i] * sc2;
      if (!inner) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // sacc[i]: key j0 + 4 quad + i, query 16 t + c16
          const int j = j0 + 4 * quad + i;
          if ((j < my_lo[t] && j >= keep) || j > my_p[t]) sv[i] = -INFINITY;
        }
      }
      const float tmax = xor32_max_f(xor16_max(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3]))));
      const float mn = fmaxf(m[t], tmax);
      const float mb = mn == -INFINITY ? 0.f : mn;  // no live key yet: exp2(-inf - 0) = 0
      alpha[t] = __builtin_amdgcn_exp2f(m[t] - mb);
      float ps = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pv = __builtin_amdgcn_exp2f(sv[i] - mb);
        ps += pv;
        pb[t][i] = (short)f2bf(pv);
      }
      ps = xor32_sum_f(xor16_sum(ps));
      l[t] = l[t] * alpha[t] + ps;
      m[t] = mn;
      rescale[t] = __any(alpha[t] != 1.f);
    }
    // wave-uniform: once the running maxima settle, most tiles skip the rescale.  ONE block for a
    // row tile's whole accumulator: a branch around each value tile's four multiplies is flattened by
    // the compiler into multiplies on every tile
#pragma unroll
    for (int t = 0; t < QT; ++t)
      if (CAP != 2 && rescale[t]) {
#pragma unroll
        for (int dt = 0; dt < DV / 16; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[t][dt][i] *= alpha[t];
      }
#pragma unroll
    for (int dt = 0; dt < DV / 16; ++dt) {
      const s16x4 a = vf[dt];
#pragma unroll
      for (int t = 0; t < QT; ++t) oacc[t][dt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, pb[t], oacc[t][dt], 0, 0, 0);
    }
   }
  }
  if (SHARED) loads_left<0>();  // none may land after the workgroup's end
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    if (CAP == 2) l[t] = xor32_sum_f(xor16_sum(l[t]));
    if (!q_live[t]) continue;  // oacc[t][dt][i] = O[q = 16 t + c16][d = 16 dt + 4 quad + i]
    float inv = l[t] > 0.f ? 1.f / l[t] : 0.f;
    if (gate != nullptr && !by_value) inv *= sigmoid_f(bf2f(gate[(long)(row0 + 16 * t + c16) * g_stride + h]));
    const bf16_t* gv = by_value ? gate + (long)(row0 + 16 * t + c16) * g_stride + (long)h * DV + 4 * quad : nullptr;
    bf16_t* orow = out + (long)(row0 + 16 * t + c16) * Hq * DV + (long)h * DV;
#pragma unroll
    for (int dt = 0; dt < DV / 16; ++dt) {
      uint2 w;
      w.x = pack2(oacc[t][dt][0] * inv, oacc[t][dt][1] * inv);
      w.y = pack2(oacc[t][dt][2] * inv, oacc[t][dt][3] * inv);
      if (by_value) w = gate_rounded(w, *reinterpret_cast<const uint2*>(gv + 16 * dt));
      *reinterpret_cast<uint2*>(orow + 16 * dt + 4 * quad) = w;
    }
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

int k8sllm_hy_window_flash(void* out, const void* qkv, long q_stride, const void* k_cache, const void* v_cache, const int* cu,
                           const int* ctx, const int* block_tables, int bt_stride, int S, long T, int Hq, int G, int dk, int dv,
                           float scale, int window, int chunked, int keep, float cap, int plain_cap, int sink,
                           const float* sinks, const void* gate, long g_stride, int by_value, hipStream_t s);
int k8sllm_hy_window_f32(void* out, const void* qkv, long q_stride, const void* k_cache, const void* v_cache, const int* cu,
                         const int* ctx, const int* block_tables, int bt_stride, int S, long T, int Hq, int G, int dk, int dv,
                         int bs, float scale, int window, int chunked, int keep, float cap, int sink, const float* sinks,
                         const void* gate, long g_stride, int decode, hipStream_t s);

int k8sllm_hy_qk_norm_cache(void* qkv, long stride, const float* qw, const float* kw, float eps, long T, int nq,
                            int nk, int nv, void* k_cache, void* v_cache, const int* slots, int bs, int singles, int f32,
                            hipStream_t s) {
  if (T <= 0) return 0;
  const int runs =
      !singles && !f32 && k_cache != nullptr && value_runs_ok(qkv, stride, nq + nk, nv, v_cache, slots, T, bs) ? value_groups(T, nv) : 0;
  const unsigned grid = (unsigned)(T + runs);
#define K8SLLM_QK(T_, NV)                                                                                             \
  hipLaunchKernelGGL((qk_norm_cache_kernel<T_, NV>), dim3(grid), dim3(256), 0, s, (T_*)qkv, stride, qw, kw, eps, nq, nk, nv, \
                     (T_*)k_cache, (T_*)v_cache, slots, bs, T, runs)
#define K8SLLM_QKT(T_)                                          \
  if (nq <= 2048 && nk <= 2048) K8SLLM_QK(T_, 8);               \
  else if (nq <= 4096 && nk <= 4096) K8SLLM_QK(T_, 16);         \
  else K8SLLM_QK(T_, 0)
  if (f32) { K8SLLM_QKT(float); } else { K8SLLM_QKT(bf16_t); }
#undef K8SLLM_QKT
#undef K8SLLM_QK
  return (int)hipGetLastError();
}

int k8sllm_hy_window_prefill(void* out, const void* qkv, long q_stride, const void* k_cache, const void* v_cache,
                             const int* cu, const int* ctx, const int* block_tables, int bt_stride, int S, long T,
                             int Hq, int G, int dk, int dv, int bs, float scale, int window, int chunked, int keep,
                             float cap, int sink, const float* sinks, const void* gate, long g_stride, int* by_value_, int f32,
                             int mfma, hipStream_t s) {
  const int by_value = *by_value_;
  if (T <= 0 || S <= 0) return 0;
  if (keep < 0 || (keep > 0 && (chunked || window <= 0))) return -1;
  if (dk > kGenDK || dv > 64 * kGenVC || G < 1 || Hq % G) return -1;
  // bf16 with matrix-core head sizes and 16-byte aligned rows: the MFMA kernel
  if (!f32 && mfma && bs == 16 && q_stride % 8 == 0 && (dk == 64 || dk == 128) && (dv == 64 || dv == 128)) {
    const long keys = window > 0 && window < 16l * bt_stride ? window : 16l * bt_stride;  // at most, per row
    if (mfma == kFlashForced || (mfma == 1 && (T * Hq >= kFlashPairs || keys >= kFlashKeys))) {
      const int rc = k8sllm_hy_window_flash(out, qkv, q_stride, k_cache, v_cache, cu, ctx, block_tables, bt_stride, S, T, Hq, G,
                                            dk, dv, scale, window, chunked, keep, cap, cap <= kMaxCapPlain && !sink, sink,
                                            sinks, gate, g_stride, by_value, s);
      if (rc != 1 || mfma == kFlashForced) return rc;
    }
    // query rows per wave: 32 once the step is large enough to fill the chip that way (two row tiles share every K / V^T
    // fragment), else 16; mfma = 16 / 32 / 64 forces one (tests, measurements).  With 32 rows four heads of one kv head,
    // where it has them, share the keys and values through LDS, and that pays from fewer (row, head) pairs.  16 rows -> 32
    // rows shared, us, 8 heads over 2 kv heads: 16384 pairs 45 -> 57 and 28 -> 33; 26000 (13 x 250) 22.0 -> 20.4; 32768
    // 75 -> 61; 52000 (13 x 500) 64 -> 40; 64000 behind 2800 keys 199 -> 90.
    const bool share = Hq / G % 4 == 0;
    const int qrows = mfma >= 16 ? mfma : (T * Hq >= (share ? 24 : 64) * 1024 ? 32 : 16);
    const int wh = share && qrows == 32 ? 4 : 0;
    const dim3 grid((unsigned)(T / qrows + S), (unsigned)(wh ? Hq / wh : Hq));
#define K8SLLM_WPC(DK, DV, QT, CAP)                            \
  if (wh && QT == 2) K8SLLM_WPW(DK, DV, 2, CAP, 4);            \
  else K8SLLM_WPW(DK, DV, QT, CAP, 0)
#define K8SLLM_WPW(DK, DV, QT, CAP, WH)                                                                                \
  hipLaunchKernelGGL((window_prefill_mfma_kernel<DK, DV, QT, CAP, WH>), grid, dim3(WH ? 64 * WH : 64), 0, s, (bf16_t*)out, \
                     (const bf16_t*)qkv, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, cu, ctx,             \
                     block_tables, bt_stride, S, Hq, G, scale, window, chunked, keep, cap, sink, sinks, (const bf16_t*)gate, g_stride, by_value)
#define K8SLLM_WP(DK, DV, QT) \
  if (cap > 0.f && cap <= kMaxCapPlain && !sink) { K8SLLM_WPC(DK, DV, QT, 2); } \
  else if (cap > 0.f) { K8SLLM_WPC(DK, DV, QT, 1); } \
  else { K8SLLM_WPC(DK, DV, QT, 0); }
#define K8SLLM_WPQ(DK, DV)                                       \
  if (qrows == 64) { K8SLLM_WP(DK, DV, 4); }                     \
  else if (qrows == 32) { K8SLLM_WP(DK, DV, 2); }                \
  else { K8SLLM_WP(DK, DV, 1); }
    if (mfma >= 16 && mfma != 16 && mfma != 32 && mfma != 64) return -1;
    if (dk == 64 && dv == 64) { K8SLLM_WPQ(64, 64); }
    else if (dk == 64) { K8SLLM_WPQ(64, 128); }
    else if (dv == 64) { K8SLLM_WPQ(128, 64); }
    else { K8SLLM_WPQ(128, 128); }
#undef K8SLLM_WPQ
#undef K8SLLM_WP
#undef K8SLLM_WPC
#undef K8SLLM_WPW
    return (int)hipGetLastError();
  }
  if (mfma == kFlashForced) return 1;
  if (by_value) gate = nullptr, *by_value_ = 0;  // (the caller gates the rows)
  if (f32 && mfma) {  // head sizes of 64 and 128: window_f32.hip, faster at every size measured there
    const int rc = k8sllm_hy_window_f32(out, qkv, q_stride, k_cache, v_cache, cu, ctx, block_tables, bt_stride, S, T, Hq, G, dk, dv,
                                        bs, scale, window, chunked, keep, cap, sink, sinks, gate, g_stride, 0, s);
    if (rc != 1) return rc;
  }
  if (f32)
    hipLaunchKernelGGL(window_prefill_kernel<float>, dim3(T, Hq), dim3(64), 0, s, (float*)out, (const float*)qkv,
                       q_stride, (const float*)k_cache, (const float*)v_cache, cu, ctx, block_tables, bt_stride, S, Hq,
                       G, dk, dv, bs, scale, window, chunked, keep, cap, sink, sinks, (const float*)gate, g_stride);
  else
    hipLaunchKernelGGL(window_prefill_kernel<bf16_t>, dim3(T, Hq), dim3(64), 0, s, (bf16_t*)out, (const bf16_t*)qkv,
                       q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, cu, ctx, block_tables, bt_stride, S,
                       Hq, G, dk, dv, bs, scale, window, chunked, keep, cap, sink, sinks, (const bf16_t*)gate, g_stride);
  return (int)hipGetLastError();
}

int k8sllm_hy_window_decode(void* out, const void* qkv, long q_stride, const void* k_cache, const void* v_cache,
                            const int* block_tables, int bt_stride, const int* seq_lens, int B, int Hq, int G, int dk,
                            int dv, int bs, float scale, int window, int chunked, int keep, float cap, int sink,
                            const float* sinks, const void* gate, long g_stride, int* by_value_, int f32, int vec, int heads,
                            hipStream_t s) {
  const int by_value = *by_value_;
  if (B <= 0) return 0;
  if (keep < 0 || (keep > 0 && (chunked || window <= 0))) return -1;
  if (dk > kGenDK || dv > 64 * kGenVC || G < 1 || Hq % G) return -1;
  const int R = Hq / G;
  const bool lanes = !f32 && vec && bs == 16 && dk % 8 == 0 && q_stride % 8 == 0 && dk <= kMaxDK && dv <= 64 * kMaxVC &&
                     (R == 1 || R == 2 || R == 4 || R == 8);
  const bool rows = lanes && (dk == 64 || dk == 128) && (dv == 64 || dv == 128);
  if (heads != 0 && (!rows || heads < 1 || R % heads || (R == 8 && heads == 4))) return -1;
  if (lanes) {
#define K8SLLM_WDR(RR, NW, ...)                                                                                        \
  hipLaunchKernelGGL((window_decode_row_kernel<RR, NW, __VA_ARGS__>), dim3(B, Hq / RR), dim3(64 * NW), 0, s, (bf16_t*)out, \
                     (const bf16_t*)qkv, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, bt_stride, \
                     seq_lens, Hq, G, scale, window, chunked, keep, cap, sink, sinks, (const bf16_t*)gate, g_stride, by_value)
#define K8SLLM_WDD(DKC, VC)                                 \
  if (R == 8 && heads == 8) K8SLLM_WDR(8, 4, DKC, VC);      \
  else if (R == 8 && heads == 2) K8SLLM_WDR(2, 4, DKC, VC); \
  else if (R == 8) K8SLLM_WDR(1, 4, DKC, VC);               \
  else if (heads == 4 && DKC + VC == 2 && (long)B * Hq > 4 * 256) K8SLLM_WDR(4, 8, DKC, VC, (DKC + VC == 2 ? 2 : 1)); \
  else if (heads == 4) K8SLLM_WDR(4, 8, DKC, VC);           \
  else if (heads == 2) K8SLLM_WDR(2, 8, DKC, VC);           \
  else K8SLLM_WDR(1, 8, DKC, VC)
    if (rows) {
      if (heads == 0) heads = decode_heads(B, Hq, R);
      if (dk == 64 && dv == 64) { K8SLLM_WDD(1, 1); }
      else if (dk == 64) { K8SLLM_WDD(1, 2); }
      else if (dv == 64) { K8SLLM_WDD(2, 1); }
      else { K8SLLM_WDD(2, 2); }
      return (int)hipGetLastError();
    }
#undef K8SLLM_WDD
#undef K8SLLM_WDR
  }
  if (by_value) gate = nullptr, *by_value_ = 0;  // (the caller gates the rows)
  if (lanes) {
#define K8SLLM_WD(RR)                                                                                                  \
  hipLaunchKernelGGL((window_decode_vec_kernel<RR, (RR == 8 ? 4 : 8)>), dim3(B, G), dim3(RR == 8 ? 256 : 512), 0, s,     \
                     (bf16_t*)out, (const bf16_t*)qkv,                                                                  \
                     q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, bt_stride, seq_lens, Hq, G, \
                     dk, dv, scale, window, chunked, keep, cap, sink, sinks, (const bf16_t*)gate, g_stride)
    if (R == 1) K8SLLM_WD(1);
    else if (R == 2) K8SLLM_WD(2);
    else if (R == 4) K8SLLM_WD(4);
    else K8SLLM_WD(8);
#undef K8SLLM_WD
    return (int)hipGetLastError();
  }
  if (f32 && vec) {
    const int rc = k8sllm_hy_window_f32(out, qkv, q_stride, k_cache, v_cache, nullptr, seq_lens, block_tables, bt_stride, B, B, Hq, G,
                                        dk, dv, bs, scale, window, chunked, keep, cap, sink, sinks, gate, g_stride, 1, s);
    if (rc != 1) return rc;
  }
  if (f32)
    hipLaunchKernelGGL(window_decode_kernel<float>, dim3(B, Hq), dim3(64), 0, s, (float*)out, (const float*)qkv,
                       q_stride, (const float*)k_cache, (const float*)v_cache, block_tables, bt_stride, seq_lens, Hq, G,
                       dk, dv, bs, scale, window, chunked, keep, cap, sink, sinks, (const float*)gate, g_stride);
  else
    hipLaunchKernelGGL(window_decode_kernel<bf16_t>, dim3(B, Hq), dim3(64), 0, s, (bf16_t*)out, (const bf16_t*)qkv,
                       q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, bt_stride, seq_lens, Hq,
                       G, dk, dv, bs, scale, window, chunked, keep, cap, sink, sinks, (const bf16_t*)gate, g_stride);
  return (int)hipGetLastError();
}
}
