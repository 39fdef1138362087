// Windowed grouped-query attention in fp32 on the fp32 matrix instruction (head sizes 64 and 128, 16-token pages); masks, sinks,
// caps and gates as in window_attn.hip, whose any-size kernel takes a wave per (row, head) and reads every key once per row.
//  * A wave has 16 query columns - prefill: 16 rows of one head; decode: the query heads of one kv head at one row - and takes a
//    page at a time: S^T[key][query] = K Q^T, then O^T[dim][query] += V^T P^T, both on v_mfma_f32_16x16x4_f32.  Both operands are
//    read as float4 along the dims (K) or the tokens (V), the quarter of a wave choosing which four; the instruction's k slots
//    are the quarters, so the float4's elements are four instructions and no data changes lanes: a lane's four scores (keys
//    4 quarter ..) are the four P operands its quarter needs.  Maxima and sums cross lanes twice (v_permlane swaps).
//  * The next page's K and V are in flight while one is processed; nothing goes through LDS but the decode merge.
//  * Decode: 8 waves take every eighth visible page and meet in LDS.
// Everything is fp32 with the any-size kernel's expf / tanhf.  A key that a query does not see is selected away before the
// softmax, and value columns past the last visible token (a page's unused end) count as zero.  An infinity or NaN among the
// values reaches the queries that see its token and no others, as there: a page that only some of a wave's queries see whole is
// looked through for one, and such values are added one by one (the matrix instruction would multiply them by the others' zeros).
// Prompts of 2 x 2048 tokens, 16 heads on 4 of 128: 13.9 -> 0.45 ms; 3 prompts of 250 to 400, 8 heads on 2: 488 -> 80 us (host
// work of the call included); decode of 2 sequences at 2048: 351 -> 31 us, of 8 at 301: 107 -> 15.  Distance to 64 bits 6.3e-7 ->
// 4.5e-7 (decode 7.1e-7 -> 3.2e-7).
#include "chunk_seg.h"

namespace k8sllm {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// max over the lanes of a query column (its four quarters)
__device__ __forceinline__ float quarters_max(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

template <int DK, int DV, bool DECODE>
__global__ __launch_bounds__(DECODE ? 512 : 64, DECODE ? 1 : 2) void window_f32_kernel(
    float* __restrict__ out, const float* __restrict__ qkv, long q_stride, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, const int* __restrict__ cu, const int* __restrict__ ctx,
    const int* __restrict__ block_tables, int bt_stride, int S, int Hq, int G, float scale, int window, int chunked, int keep,
    float cap, int sink, const float* __restrict__ sinks, const float* __restrict__ gate, long g_stride) {
  constexpr int NW = DECODE ? 8 : 1, KG = DK / 16, VG = DV / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, qt = lane >> 4;
  const int R = Hq / G;
  // this column's row, head and position; n columns are real
  int n, seg, row, h, p0, p;
  if (DECODE) {  // ctx: the sequences' lengths, this token included
    seg = row = blockIdx.x;
    n = R;
    h = blockIdx.y * R + min(col, R - 1);
    p0 = p = ctx[seg] - 1;
    if (p < 0) {  // padding row of a decode bucket
      for (int c = threadIdx.x; c < R * DV; c += 512) out[(long)row * Hq * DV + (long)blockIdx.y * R * DV + c] = 0.f;
      return;
    }
  } else {
    const ChunkAt at = chunk_at(cu, S, blockIdx.x, 16);
    if (at.seg < 0) return;
    seg = at.seg;
    n = at.n;
    h = blockIdx.y;
    p0 = ctx[seg] + 16 * at.k;
    p = p0 + min(col, n - 1);
    row = at.row + min(col, n - 1);
  }
  const int g = h / R, hi = DECODE ? p + 1 : p0 + n;  // no column sees a position from hi on
  const int lo = first_key(p, window, chunked);
  const int lo_last = DECODE ? lo : first_key(p0 + n - 1, window, chunked);  // from here to p0: keys that every column sees
  // pages: the kept ones, then those from the first column's window on
  const int w_first = first_key(p0, window, chunked) >> 4, k_end = (keep + 15) >> 4;
  const int t_end = (hi + 15) >> 4, gap_from = keep > 0 ? k_end : 0, gap_to = max(w_first, gap_from);
  const int tiles = min(gap_from, t_end) + max(t_end - gap_to, 0);
  auto page_of = [&](int i) { return i < gap_from ? i : i - gap_from + gap_to; };
  const int* bt = block_tables + (long)seg * bt_stride;
  f32x4 q[KG];
  {
    const float* qp = qkv + (long)row * q_stride + (long)h * DK + 4 * qt;
#pragma unroll
    for (int i = 0; i < KG; ++i) q[i] = *reinterpret_cast<const f32x4*>(qp + 16 * i) * scale;
  }
  const float sink_z = sink && sinks != nullptr ? sinks[h] : 0.f;
  const bool has_sink = sink && qt == 0 && wave == 0;  // counted once
  float m = sink ? sink_z : -INFINITY, l = has_sink ? 1.f : 0.f;
  f32x4 o[VG] = {};
  f32x4 kn[KG], vn[VG];
  auto load = [&](int i) {
    const long page = bt[page_of(i)];
    const float* kp = k_cache + ((page * 16 + col) * G + g) * DK + 4 * qt;
    const float* vp = v_cache + ((page * G + g) * DV + col) * 16 + 4 * qt;
#pragma unroll
    for (int u = 0; u < KG; ++u) kn[u] = *reinterpret_cast<const f32x4*>(kp + 16 * u);
#pragma unroll
    for (int u = 0; u < VG; ++u) vn[u] = *reinterpret_cast<const f32x4*>(vp + 256 * u);
  };
  if (wave < tiles) load(wave);
  for (int i = wave; i < tiles; i += NW) {
    f32x4 k[KG], v[VG];
#pragma unroll
    for (int u = 0; u < KG; ++u) k[u] = kn[u];
#pragma unroll
    for (int u = 0; u < VG; ++u) v[u] = vn[u];
    if (i + NW < tiles) load(i + NW);
    const int key = page_of(i) * 16 + 4 * qt;  // this lane's keys (and value tokens): key .. key + 3
    f32x4 s0 = {}, s1 = {};
#pragma unroll
    for (int u = 0; u < KG; u += 2)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u][j], q[u][j], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[u + 1][j], q[u + 1][j], s1, 0, 0, 0);
      }
    f32x4 s = s0 + s1;
    float mt = m;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (cap > 0.f) s[j] = cap * tanhf(s[j] / cap);
      const int kk = key + j;
      s[j] = kk <= p && (kk >= lo || kk < keep) ? s[j] : -INFINITY;
      mt = fmaxf(mt, s[j]);
    }
    mt = quarters_max(mt);
    const float base = mt == -INFINITY ? 0.f : mt;  // nothing seen yet: every term is 0
    const float alpha = expf(m - base);
    m = mt;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[j] = expf(s[j] - base);
      sum += s[j];
    }
    l = l * alpha + sum;
    if (key + 3 >= hi) {
#pragma unroll
      for (int u = 0; u < VG; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[u][j] = key + j < hi ? v[u][j] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < VG; ++u) o[u] *= alpha;
    const int k0 = page_of(i) * 16;
    if (k0 + 15 > p0 || (k0 < lo_last && k0 + 15 >= keep)) {  // wave-uniform
      float z = 0.f;  // NaN if any value is no number
#pragma unroll
      for (int u = 0; u < VG; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) z = fmaf(v[u][j], 0.f, z);
      if (__any(z != z)) {
#pragma unroll 1
        for (int a = 0; a < 4; ++a)  // tokens k0 + 4 a + j
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int kk = k0 + 4 * a + j;
            const float w = __shfl(s[j], 16 * a + col);
            const bool seen = kk <= p && (kk >= lo || kk < keep);
#pragma unroll
            for (int u = 0; u < VG; ++u)
#pragma unroll
              for (int d = 0; d < 4; ++d) {
                const float x = __shfl(v[u][j], 16 * a + 4 * qt + d);
                if (seen && !isfinite(x)) o[u][d] = fmaf(w, x, o[u][d]);
              }
          }
#pragma unroll
        for (int u = 0; u < VG; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j) v[u][j] = isfinite(v[u][j]) ? v[u][j] : 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int u = 0; u < VG; ++u) o[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[u][j], s[j], o[u], 0, 0, 0);
  }
  l = xor32_sum_f(xor16_sum(l));
  const float gt = gate != nullptr ? sigmoid_f(gate[(long)row * g_stride + h]) : 1.f;
  if (DECODE) {  // the waves' parts: maxima and sums, then the outputs one dim group at a time
    __shared__ float ms[NW][16], ls[NW][16];
    __shared__ __attribute__((aligned(16))) float os[NW][8][DV + 4];
    if (qt == 0) {
      ms[wave][col] = m;
      ls[wave][col] = l;
    }
    if (col < 8)
#pragma unroll
      for (int u = 0; u < VG; ++u) *reinterpret_cast<f32x4*>(&os[wave][col][16 * u + 4 * qt]) = o[u];
    __syncthreads();
    for (int i = threadIdx.x; i < R * DV; i += 512) {
      const int c = i / DV, d = i % DV;
      float mm = ms[0][c], ll = 0.f, a = 0.f;
#pragma unroll
      for (int w = 1; w < NW; ++w) mm = fmaxf(mm, ms[w][c]);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float f = ms[w][c] == -INFINITY ? 0.f : expf(ms[w][c] - mm);
        ll += f * ls[w][c];
        a += f * os[w][c][d];
      }
      const int hh = blockIdx.y * R + c;
      const float gg = gate != nullptr ? sigmoid_f(gate[(long)row * g_stride + hh]) : 1.f;
      out[(long)row * Hq * DV + (long)hh * DV + d] = ll > 0.f ? a * (gg / ll) : 0.f;
    }
  } else if (col < n) {
    const float inv = l > 0.f ? gt / l : 0.f;
    float* op = out + (long)row * Hq * DV + (long)h * DV + 4 * qt;
#pragma unroll
    for (int u = 0; u < VG; ++u) *reinterpret_cast<f32x4*>(op + 16 * u) = o[u] * inv;
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

// T rows of S segments (decode: B = S rows, ctx their lengths).  1: not these sizes
int k8sllm_hy_window_f32(void* out, const void* qkv, long q_stride, const void* k_cache, const void* v_cache, const int* cu,
                         const int* ctx, const int* block_tables, int bt_stride, int S, long T, int Hq, int G, int dk, int dv,
                         int bs, float scale, int window, int chunked, int keep, float cap, int sink, const float* sinks,
                         const void* gate, long g_stride, int decode, hipStream_t s) {
  if (bs != 16 || (dk != 64 && dk != 128) || (dv != 64 && dv != 128) || q_stride % 4 != 0) return 1;
  if (decode && Hq / G > 8) return 1;
  if ((reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache) |
       reinterpret_cast<uintptr_t>(out)) & 15)
    return 1;
  const dim3 grid = decode ? dim3((unsigned)S, (unsigned)G) : dim3((unsigned)(T / 16 + S), (unsigned)Hq);
#define K8SLLM_WF(DK, DV, DEC)                                                                                           \
  hipLaunchKernelGGL((window_f32_kernel<DK, DV, DEC>), grid, dim3(DEC ? 512 : 64), 0, s, (float*)out, (const float*)qkv, q_stride, \
                     (const float*)k_cache, (const float*)v_cache, cu, ctx, block_tables, bt_stride, S, Hq, G, scale, window,     \
                     chunked, keep, cap, sink, sinks, (const float*)gate, g_stride)
#define K8SLLM_WFD(DEC)                                        \
  if (dk == 64 && dv == 64) K8SLLM_WF(64, 64, DEC);            \
  else if (dk == 64) K8SLLM_WF(64, 128, DEC);                  \
  else if (dv == 64) K8SLLM_WF(128, 64, DEC);                  \
  else K8SLLM_WF(128, 128, DEC)
  if (decode) { K8SLLM_WFD(true); } else { K8SLLM_WFD(false); }
#undef K8SLLM_WFD
#undef K8SLLM_WF
  return (int)hipGetLastError();
}
}
