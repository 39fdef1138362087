// The per-head products around latent attention for the rows of a decode step (bf16): queries into the latent space with their turned part, and
// latents to values.  They read the expansions once, a megabyte or two; what bounds them is the latency of one chain of loads, products and stores,
// so a wave takes the smallest tile that its matrix instruction fills, with its weights' loads in flight together, and the grid is as wide as that
// gives.  The library's batched products with the launch that put the rows together / these, us: queries of 8 heads of 96 + 32
// over 256, 1 row 11.6 / 4.2, 64 13.5 / 4.7, 512 14.1 / 5.8; 16 heads, 64 rows 18.9 / 4.4; values of 8 heads of 128, 1 row 7.3 / 4.5, 64 5.9 / 4.9.
#include "latent_parts.h"

namespace k8sllm {

typedef __bf16 hbf16x8 __attribute__((ext_vector_type(8)));
typedef float hf32x4 __attribute__((ext_vector_type(4)));

// v_mfma_f32_16x16x32_bf16, A's row and B's column lane & 15, eight values of k from 8 (lane >> 4); results of rows 4 (lane >> 4) + 0 .. 3
__device__ __forceinline__ hf32x4 tile_product(const uint4& a, const uint4& b, const hf32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(hbf16x8, a), __builtin_bit_cast(hbf16x8, b), c, 0, 0, 0);
}

// out[t][h] = [q[t][h][:dn] W[h] | the last dr entries of q[t][h], turned | zeros to the pitch w].  Workgroup (x, h, z), one wave: 128 columns of 16
// rows.  W[h] is [dn][R]: a lane reads eight rows' eight columns 8 (lane & 15) + j and turns them about, so that product j has columns 8 i + j
// and a lane's results are 32 neighbouring columns.  The last four x: the rest of four rows each.
__global__ __launch_bounds__(64) void latent_head_queries_kernel(bf16_t* __restrict__ out, const bf16_t* __restrict__ q, long q_stride,
                                                                 const bf16_t* __restrict__ wk, int T, int H, int dn, int dr, int R, int w,
                                                                 const int* __restrict__ positions, const float* __restrict__ freq, int nf,
                                                                 int pairs) {
  const int h = blockIdx.y, t0 = 16 * blockIdx.z, lane = threadIdx.x, col = lane & 15, quad = lane >> 4, nt = (R + 127) / 128;
  if (blockIdx.x >= nt) {
    const int n = w - R, r0 = t0 + 4 * (blockIdx.x - nt), nr = min(4, T - r0);
    for (int e = lane; e < nr * n; e += 64) {
      const int r = e / n, i = e - r * n;
      const long t = r0 + r;
      const bf16_t* qr = q + t * q_stride + (long)h * (dn + dr) + dn;
      bf16_t* o = out + (t * H + h) * w + R;
      if (i >= dr) {
        o[i] = 0;
      } else if (i >= 2 * nf) {
        o[i] = qr[i];
      } else if (i < nf) {  // the pair (a, b)
        const int a = pairs ? 2 * i : i, b = pairs ? 2 * i + 1 : i + nf;
        float sn, cs;
        sincosf((float)positions[t] * freq[i], &sn, &cs);
        const float u = ldf(qr + a), v = ldf(qr + b);
        stf(o + a, fmaf(u, cs, -(v * sn)));
        stf(o + b, fmaf(v, cs, u * sn));
      }
    }
    return;
  }
  const int n0 = 128 * blockIdx.x + 8 * col;
  const bf16_t* wr = wk + (long)h * dn * R + min(n0, R - 8);
  const bf16_t* qr = q + (long)min(t0 + col, T - 1) * q_stride + (long)h * (dn + dr);
  hf32x4 acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = hf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 8 * quad; k < dn + 8 * quad; k += 32) {  // (every lane takes part in each product)
    const bool in = k < dn;
    const int kc = in ? k : 0;
    uint4 b = *reinterpret_cast<const uint4*>(qr + kc), r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = *reinterpret_cast<const uint4*>(wr + (long)(kc + i) * R);
    if (!in) b = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      uint32_t f[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        uint32_t x = j < 2 ? r[2 * m].x : j < 4 ? r[2 * m].y : j < 6 ? r[2 * m].z : r[2 * m].w;
        uint32_t y = j < 2 ? r[2 * m + 1].x : j < 4 ? r[2 * m + 1].y : j < 6 ? r[2 * m + 1].z : r[2 * m + 1].w;
        f[m] = __builtin_amdgcn_perm(y, x, j & 1 ? 0x07060302u : 0x05040100u);
        if (!in) f[m] = 0;
      }
      acc[j] = tile_product(make_uint4(f[0], f[1], f[2], f[3]), b, acc[j]);
    }
  }
  if (t0 + col >= T) return;
  bf16_t* o = out + ((long)(t0 + col) * H + h) * w + 128 * blockIdx.x + 32 * quad;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = acc[j][i];
    if (128 * (int)blockIdx.x + 32 * quad + 8 * i < R) store8(o + 8 * i, v);
  }
}

// v[t][h] = W[h] o[t][h], W[h] [dv][R].  Workgroup (x, h, z), one wave: 16 values of 16 rows.
__global__ __launch_bounds__(64) void latent_head_values_kernel(bf16_t* __restrict__ v, const bf16_t* __restrict__ o, const bf16_t* __restrict__ wv,
                                                                int T, int H, int dv, int R) {
  const int h = blockIdx.y, t0 = 16 * blockIdx.z, lane = threadIdx.x, col = lane & 15, quad = lane >> 4, n0 = 16 * blockIdx.x;
  const bf16_t* wr = wv + ((long)h * dv + min(n0 + col, dv - 1)) * R;
  const bf16_t* orow = o + ((long)min(t0 + col, T - 1) * H + h) * R;
  hf32x4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k = 8 * quad; k < R + 8 * quad; k += 32) {
    const bool in = k < R;
    uint4 a = *reinterpret_cast<const uint4*>(wr + (in ? k : 0)), b = *reinterpret_cast<const uint4*>(orow + (in ? k : 0));
    if (!in) a = b = make_uint4(0, 0, 0, 0);
    acc = tile_product(a, b, acc);
  }
  if (t0 + col >= T) return;
  bf16_t* out = v + ((long)(t0 + col) * H + h) * dv + n0 + 4 * quad;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (n0 + 4 * quad + i < dv) stf(out + i, acc[i]);
}

// The same of rows whose attention lies in parts (LatentParts): their merge, times the sigmoid of the row and head's gate, rounded, is the products' operand.
// Each of a head's dv / 16 workgroups merges its rows again, which costs less than a launch of its own (1.6 us and a round of loads).
// NW waves take the parts in turn and put their pieces of R into LDS, and one more multiplies: in the order of latent_head_values_kernel, and rows of one
// part with what is already finished for them, so that a row has the same bits whatever stands beside it.  Sixteen rows of one part each need nothing
// else.  All that may be needed is on its way before it is known what is (a round of loads less: 64 rows of 1500 keys, 16 heads, 32.7 / 31.9 us).  Three
// waves for three parts: two workgroups of five waves share no unit (64 rows of 700 keys, 16 heads, 26.2 / 24.6).
template <int NW>
__global__ __launch_bounds__(64 * (NW + 1)) void latent_part_values_kernel(bf16_t* __restrict__ v, const bf16_t* __restrict__ one, LatentParts parts, int most,
                                                                           const bf16_t* __restrict__ wv, int T, int H, int dv, int R,
                                                                           const bf16_t* __restrict__ gate, long g_stride) {
  constexpr int KC = 8;  // pieces of 32 k: R <= 256
  __shared__ __attribute__((aligned(16))) float4 o_s[NW][2 * KC][64];
  __shared__ float2 ml_s[NW][64];
  __shared__ uint4 x_s[KC][64];
  const int h = blockIdx.y, t0 = 16 * blockIdx.z, lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // (scalar: the waves' branches hold barriers)
  const int n0 = 16 * blockIdx.x, t = min(t0 + col, T - 1);
  const long th = (long)t * H + h, step = (long)T * H;
  const int np = parts.n[t];
  if (wave == NW) {
    uint4 a[KC], b[KC];
    auto load = [&](uint4 (&x)[KC], const bf16_t* row) {
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const int k = 32 * c + 8 * quad;
        x[c] = *reinterpret_cast<const uint4*>(row + (k < R ? k : 0));
        if (k >= R) x[c] = make_uint4(0, 0, 0, 0);
      }
    };
    load(a, wv + ((long)h * dv + min(n0 + col, dv - 1)) * R);
    load(b, one + th * R);
    if (__ballot(np > 1) != 0) {  // the same rows in every wave
      __syncthreads();
      __syncthreads();
      if (np > 1) {
#pragma unroll
        for (int c = 0; c < KC; ++c)
          if (32 * c + 8 * quad < R) b[c] = x_s[c][lane];
      }
    }
    hf32x4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KC; ++c)
      if (32 * c < R) acc = tile_product(a[c], b[c], acc);
    if (t0 + col >= T) return;
    bf16_t* out = v + ((long)(t0 + col) * H + h) * dv + n0 + 4 * quad;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n0 + 4 * quad + i < dv) stf(out + i, acc[i]);
    return;
  }
  float2 ml;
  float x[KC][8];
  auto part = [&](int z) {  // (what is not there is in the buffer, and read by nobody)
    const long at = z < most ? z * step + th : 0;
    const float* p = parts.o + at * R + 8 * quad;
    ml = parts.ml[at];
#pragma unroll
    for (int c = 0; c < KC; ++c) load8(p + (32 * c + 8 * quad < R ? 32 * c : -8 * quad), x[c]);
  };
  part(wave);
  if (__ballot(np > 1) == 0) return;
  float M = -INFINITY, L = 0.f, o[KC][8] = {};
  for (int z = wave; __ballot(np > 1 && z < np) != 0; z += NW) {
    if (z > wave) part(z);
    if (np <= 1 || z >= np) continue;
    const float m = fmaxf(M, ml.x), f0 = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - m), f1 = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - m);
    M = m;
    L = fmaf(ml.y, f1, L * f0);
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) o[c][j] = fmaf(x[c][j], f1, o[c][j] * f0);
  }
#pragma unroll
  for (int c = 0; c < KC; ++c) {
    o_s[wave][2 * c][lane] = make_float4(o[c][0], o[c][1], o[c][2], o[c][3]);
    o_s[wave][2 * c + 1][lane] = make_float4(o[c][4], o[c][5], o[c][6], o[c][7]);
  }
  ml_s[wave][lane] = make_float2(M, L);
  __syncthreads();
  float f[NW];
  M = -INFINITY;
  L = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) M = fmaxf(M, ml_s[w][lane].x);
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float2 q = ml_s[w][lane];
    f[w] = q.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(q.x - M);
    L = fmaf(q.y, f[w], L);
  }
  float inv = L > 0.f ? 1.f / L : 0.f;
  if (gate != nullptr) inv *= sigmoid_f(bf2f(gate[(long)t * g_stride + h]));
#pragma unroll
  for (int i = 0; i < (KC + NW - 1) / NW; ++i) {
    const int c = NW * i + wave;
    if (c >= KC) break;
    float y[8] = {};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float4 u = o_s[w][2 * c][lane], s = o_s[w][2 * c + 1][lane];
      const float q[8] = {u.x, u.y, u.z, u.w, s.x, s.y, s.z, s.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = fmaf(q[j], f[w], y[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] *= inv;
    x_s[c][lane] = pack8(y);
  }
  __syncthreads();
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

// -1: not these sizes (whole 16-byte pieces of rows and weights)
int k8sllm_hy_latent_head_queries(void* out, const void* q, long q_stride, const void* wk, long T, int H, int dn, int dr, int R, int w,
                                  const int* positions, const float* freq, int nf, int pairs, hipStream_t s) {
  if (T <= 0 || H <= 0) return 0;
  if (dn < 8 || R < 8 || (dn | dr | R | w) % 8 || q_stride % 8 || T > (1 << 19) || H > 65535 || w < R + dr || 2 * nf > dr ||
      ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(wk)) & 15))
    return -1;
  hipLaunchKernelGGL(latent_head_queries_kernel, dim3((unsigned)((R + 127) / 128 + (w > R ? 4 : 0)), (unsigned)H, (unsigned)((T + 15) / 16)),
                     dim3(64), 0, s, (bf16_t*)out, (const bf16_t*)q, q_stride, (const bf16_t*)wk, (int)T, H, dn, dr, R, w, positions, freq, nf,
                     pairs);
  return (int)hipGetLastError();
}

int k8sllm_hy_latent_head_values(void* v, const void* o, const void* wv, long T, int H, int dv, int R, hipStream_t s) {
  if (T <= 0 || H <= 0 || dv <= 0) return 0;
  if (R < 8 || R % 8 || T > (1 << 19) || H > 65535 || ((reinterpret_cast<uintptr_t>(o) | reinterpret_cast<uintptr_t>(wv)) & 15)) return -1;
  hipLaunchKernelGGL(latent_head_values_kernel, dim3((unsigned)((dv + 15) / 16), (unsigned)H, (unsigned)((T + 15) / 16)), dim3(64), 0, s,
                     (bf16_t*)v, (const bf16_t*)o, (const bf16_t*)wv, (int)T, H, dv, R);
  return (int)hipGetLastError();
}

// most: how many parts the buffers hold
int k8sllm_hy_latent_part_values(void* v, const void* one, const float* o, const void* ml, const int* n, int most, const void* wv, long T, int H,
                                 int dv, int R, const void* gate, long g_stride, hipStream_t s) {
  if (T <= 0 || H <= 0 || dv <= 0) return 0;
  if (R < 16 || R % 16 || R > 256 || T > (1 << 19) || H > 65535 || most < 1 || (reinterpret_cast<uintptr_t>(wv) & 15)) return -1;
  const dim3 grid((unsigned)((dv + 15) / 16), (unsigned)H, (unsigned)((T + 15) / 16));
  const LatentParts p{(float*)o, (float2*)ml, (int*)n, 0};
  if (most <= 3)
    hipLaunchKernelGGL(latent_part_values_kernel<3>, grid, dim3(256), 0, s, (bf16_t*)v, (const bf16_t*)one, p, most, (const bf16_t*)wv, (int)T, H, dv, R,
                       (const bf16_t*)gate, g_stride);
  else
    hipLaunchKernelGGL(latent_part_values_kernel<4>, grid, dim3(320), 0, s, (bf16_t*)v, (const bf16_t*)one, p, most, (const bf16_t*)wv, (int)T, H, dv, R,
                       (const bf16_t*)gate, g_stride);
  return (int)hipGetLastError();
}
}
