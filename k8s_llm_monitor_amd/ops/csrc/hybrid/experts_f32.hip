// Experts' fp32 products Y[r] = W[e(r)] A[row(r)] over expert-sorted rows on the bf16 matrix instruction, K a multiple of 32, rows
// 16-byte aligned.  An fp32 number is the sum of three bf16 numbers (rounded to nearest each time, the differences exact), bf16 products
// are exact, and six of the nine products of two such sums hold all of theirs but 2^-26 of it: hh, hm, mh, mm, hl, lh.  hh has sums of
// its own, so that large numbers are rounded once in 32 products: at K = 1024 2.1e-7 of the result from 64 bits, the fp32 instruction 5.7e-7.
//   Tile: 64 rows x 64 NB weight rows (gated: 64 gate and 64 up), four waves with 32 rows x 32 columns of each block.  A thread splits
//   eight k of a row of every block and stores the three parts to LDS, one step of 32 k at a time: the next step is split beside the
//   matrix instructions, its loads are a step ahead, and one slot leaves a CU three workgroups whose phases overlap (two slots
//   and two workgroups: 63.7 us for 57.7).  Chunk c of a row lies at c ^ (row / 4 % 4): the fragments' reads are spread over the
//   banks.  Bound by the matrix cores' rate under load (12.4 ns an instruction, 48 a step and wave) and the splitting beside it.
// 1772 rows over 8 experts, K = N = 1024, gated / plain: 95 / 52 us on the fp32 instruction, 58 / 39 here; 16 rows 52 / 33, 38 / 24.
// What is no number: an infinity's or NaN's parts make every result that it reaches a NaN, and a result that is a NaN is computed
// again on the vector unit, so that infinities come out as fp32 products have them.
// Operands below 2^-110 keep fewer bits, their last ones lying below bf16's denormals: rows of 2^-112 leave results 1.7e-7 off, of 2^-115 1.1e-6, of
// 2^-126 2e-3 (the fp32 instruction 3e-7 for all three; down to 2^-110 9e-8 here).  Splitting 2^24 times the operands keeps every bit and took
// 1024 x 1024 beside 8 experts from 28.5 to 34.1 us for 16 rows, from 118 to 122 for 8000.
#include "split_bf16.h"

namespace k8sllm {

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t round2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// eight values' three parts
__device__ __forceinline__ void split8(const float4& a, const float4& b, uint4 (&p)[3]) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    h[i] = round2(x[2 * i], x[2 * i + 1]);
    const float r0 = x[2 * i] - lo_bf(h[i]), r1 = x[2 * i + 1] - hi_bf(h[i]);
    m[i] = round2(r0, r1);
    l[i] = round2(r0 - lo_bf(m[i]), r1 - hi_bf(m[i]));
  }
  p[0] = make_uint4(h[0], h[1], h[2], h[3]);
  p[1] = make_uint4(m[0], m[1], m[2], m[3]);
  p[2] = make_uint4(l[0], l[1], l[2], l[3]);
}

__device__ __forceinline__ float gelu_erf_f32(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }

}  // namespace

struct ExpertsF32 {
  float* y;
  const float* a;
  const float* w;
  const int* offsets;     // expert e's rows are offsets[e] .. offsets[e + 1] - 1
  const int* sorted_idx;  // row r is row sorted_idx[r] / div of a; null: row r
  long w_es;
  int div, E, N, Kd, il;
  float limit;
};

// ACT as in moe_ffn.hip: 0 none, 1 SwiGLU, 2 erf GELU, 3 the clamped unit, 4 squared ReLU
template <int ACT, int NB>
__global__ __launch_bounds__(256, 3) void experts_f32_kernel(ExpertsF32 g) {
  constexpr bool GATED = ACT == 1 || ACT == 3;
  static_assert(!GATED || NB == 2, "");
  constexpr int PLANE = (1 + NB) * 64 * 64, TK = 32;  // bytes of one part: the rows' 64, then the weights' 64 NB, of 64 bytes each
  __shared__ __attribute__((aligned(1024))) char buf[3 * PLANE];
  int e, tile = blockIdx.y, r0, r1;
  if (!expert_tile<64>(g.offsets, g.E, tile, e, r0, r1)) return;
  r0 += tile * 64;
  const int n0 = blockIdx.x * (GATED ? 64 : 64 * NB);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, quad = lane >> 4, wm = wave & 1, wn = wave >> 1;
  auto arow = [&](int r) { return g.a + (long)(g.sorted_idx != nullptr ? g.sorted_idx[r] / g.div : r) * g.Kd; };
  auto wrow = [&](int b, int n) {  // row of W behind column n of block b
    const long gate = GATED && g.il ? (long)(n >> 6) * 128 + (n & 63) : n;
    return g.w + (long)e * g.w_es + (GATED && b ? (g.il ? gate + 64 : (long)g.N + n) : gate) * g.Kd;
  };
  auto col = [&](int b, int j) { return n0 + (GATED ? 0 : 64 * b) + j; };
  const int srow = threadIdx.x >> 2, sch = threadIdx.x & 3;
  const float* src[1 + NB];
  src[0] = arow(min(r0 + srow, r1 - 1)) + 8 * sch;
#pragma unroll
  for (int b = 0; b < NB; ++b) src[1 + b] = wrow(b, min(col(b, srow), g.N - 1)) + 8 * sch;
  const int sto = srow * 64 + ((sch ^ ((srow >> 2) & 3)) << 4);
  const int nk = g.Kd / TK;
  float4 v[1 + NB][2];
  auto load = [&](int k) {  // steps past the last repeat it; nothing multiplies them
#pragma unroll
    for (int q = 0; q < 1 + NB; ++q)
#pragma unroll
      for (int i = 0; i < 2; ++i) v[q][i] = *reinterpret_cast<const float4*>(src[q] + TK * min(k, nk - 1) + 4 * i);
  };
  uint4 p[1 + NB][3];
  auto split = [&]() {
#pragma unroll
    for (int q = 0; q < 1 + NB; ++q) split8(v[q][0], v[q][1], p[q]);
  };
  auto store = [&]() {
#pragma unroll
    for (int q = 0; q < 1 + NB; ++q)
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(buf + i * PLANE + q * 4096 + sto) = p[q][i];
  };
  f32x4 acc[NB][2][2] = {}, low[NB][2][2] = {};  // hh; the other five, so that the large sums are rounded once a step
  const int rd = c16 * 64 + ((quad ^ (c16 >> 2)) << 4);
  auto frag = [&](int part, int row) { return *reinterpret_cast<const bf16x8*>(buf + part * PLANE + row * 64 + rd); };
  load(0);
  split();
  load(1);
  for (int k = 0; k < nk; ++k) {
    lds_barrier();  // the last step's parts have been read
    store();
    lds_barrier();  // this step's parts are there
    bf16x8 a[2][3], w[2][3];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) a[i][p] = frag(p, wm * 32 + 16 * i);
    split();  // the next step's
    load(k + 2);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int p = 0; p < 3; ++p) w[j][p] = frag(p, 64 + 64 * u + wn * 32 + 16 * j);
      constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PW[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            f32x4& c = t < 5 ? low[u][i][j] : acc[u][i][j];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][PA[t]], w[j][PW[t]], c, 0, 0, 0);
          }
    }
  }
#pragma unroll
  for (int u = 0; u < NB; ++u)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[u][i][j] += low[u][i][j];
  auto value = [&](float z, int r, int b, int n) {
    if (z == z) return z;
    const float* x = arow(r);
    const float* y = wrow(b, n);
    z = 0.f;
    for (int k = 0; k < g.Kd; ++k) z = fmaf(x[k], y[k], z);
    return z;
  };
#pragma unroll
  for (int u = 0; u < (GATED ? 1 : NB); ++u)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = col(u, wn * 32 + 16 * j + c16);
      if (n >= g.N) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = r0 + wm * 32 + 16 * i + 4 * quad + q;
          if (r >= r1) continue;
          float z = value(acc[u][i][j][q], r, u, n);
          if (ACT == 1) z = silu_f(z) * value(acc[NB - 1][i][j][q], r, 1, n);
          if (ACT == 3) {
            const float gt = fminf(z, g.limit), up = fminf(fmaxf(value(acc[NB - 1][i][j][q], r, 1, n), -g.limit), g.limit);
            z = gt * sigmoid_f(1.702f * gt) * (up + 1.f);
          }
          if (ACT == 2) z = gelu_erf_f32(z);
          if (ACT == 4) z = z > 0.f ? z * z : 0.f;
          g.y[(long)r * g.N + n] = z;
        }
    }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

int k8sllm_hy_experts_f32(float* y, const float* a, const float* w, const int* offsets, const int* sorted_idx, int div, int E, long rows,
                          int N, int Kd, long w_es, int act, int il, float limit, hipStream_t s) {
  if (rows <= 0 || N <= 0) return 0;
  if (act < 0 || act > 4 || Kd < 32 || Kd % 32 || ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15)) return -1;
  const bool gated = act == 1 || act == 3;
  const ExpertsF32 g{y, a, w, offsets, sorted_idx, w_es, div, E, N, Kd, il, limit};
  // 64 columns a workgroup until 128 leave every CU one (N = 1024: 1772 rows 39 / 46 us, 1996 53 / 48, 3000 62 / 54)
  const unsigned mt = (unsigned)(rows / 64 + E);
  const int nb = gated || (long)mt * ((N + 127) / 128) >= 300 ? 2 : 1;
  const int cols = gated ? 64 : 64 * nb;
  const dim3 grid((unsigned)((N + cols - 1) / cols), mt);  // consecutive column tiles: an expert's row tiles meet them in the same L2
#define K8SLLM_XF(ACT, NB) hipLaunchKernelGGL((experts_f32_kernel<ACT, NB>), grid, dim3(256), 0, s, g)
#define K8SLLM_XFP(ACT) \
  if (nb == 2) K8SLLM_XF(ACT, 2); \
  else K8SLLM_XF(ACT, 1)
  if (act == 1) K8SLLM_XF(1, 2);
  else if (act == 3) K8SLLM_XF(3, 2);
  else if (act == 2) { K8SLLM_XFP(2); }
  else if (act == 4) { K8SLLM_XFP(4); }
  else { K8SLLM_XFP(0); }
#undef K8SLLM_XFP
#undef K8SLLM_XF
  return (int)hipGetLastError();
}
}
