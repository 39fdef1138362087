// Y[M][N] = X[M][K] W[N][K]^T for the few rows of a decode step (bf16, fp32 sums, M up to 64, K a multiple of 32).
// A projection of a few rows is a pass over its weights; what a call takes is set by how soon enough loads are in flight, and by how
// often the rows are fetched beside the weights.  Two forms (stream_rows.h has the streams):
//   own     a workgroup takes 16 columns, its four waves a quarter of K each with their own copies of the rows; the waves' sums meet in
//           LDS in the order of K.  As many workgroups as there are column tiles.
//   shared  a workgroup takes 64 columns and all of K, its four waves share the rows.
#include "stream_rows.h"

namespace k8sllm {

// What becomes of a product: KIND -1 nothing; 1, 3, 4: W's first 2 f rows are a gated unit's gate and up rows, Yg [M][f] = act(gate) * up of
// the products rounded to bf16 (as the separate launch finds them), Y gets the products of the rest; 16 + a: act_f<a> of the rounded
// product.  One launch less each.  F32: Y is fp32, the rounded products capped at +-cap if cap > 0 (logits).
struct RowsOut {
  void* y;
  bf16_t* yg;
  int M, N, f, f32;
  float cap;
};

template <int KIND>
__device__ __forceinline__ void rows_store(const RowsOut& o, int r, int n, float v) {  // n: row of W
  if (r >= o.M || n >= o.N) return;
  const int first = KIND >= 0 && KIND < 16 ? 2 * o.f : 0;
  const long i = (long)r * (o.N - first) + n - first;
  const bf16_t b = f2bf(v);
  if (KIND >= 16) {
    reinterpret_cast<bf16_t*>(o.y)[i] = f2bf(act_f<KIND >= 16 ? KIND - 16 : 3>(bf2f(b), 0.f, 0.f));
  } else if (o.f32) {
    const float z = bf2f(b);
    reinterpret_cast<float*>(o.y)[i] = o.cap > 0.f ? o.cap * tanhf(z / o.cap) : z;
  } else {
    reinterpret_cast<bf16_t*>(o.y)[i] = b;
  }
}
template <int KIND>
__device__ __forceinline__ void rows_store_unit(const RowsOut& o, int r, int n, float g, float u) {
  if (r < o.M) o.yg[(long)r * o.f + n] = f2bf(glu_unit<KIND >= 0 && KIND < 16 ? KIND : 3>(bf2f(f2bf(g)), bf2f(f2bf(u)), 0.f));
}

// Column tile ``j`` of a launch: gated kinds take two tiles of W's rows, a unit's gate and up or two neighbours of the rest
template <int KIND>
__device__ __forceinline__ bool rows_tiles(int j, int f, int (&n)[KIND >= 0 && KIND < 16 ? 2 : 1]) {
  if constexpr (KIND >= 0 && KIND < 16) {
    const bool pair = j < f / 16;
    n[0] = pair ? 16 * j : 2 * f + 32 * (j - f / 16);
    n[1] = pair ? n[0] + f : n[0] + 16;
    return pair;
  } else {
    n[0] = 16 * j;
    return false;
  }
}

template <int KIND, int MT, bool ONCE>
__global__ __launch_bounds__(256) void few_rows_own_kernel(RowsOut o, const bf16_t* __restrict__ X, long x_stride,
                                                           const bf16_t* __restrict__ W, int Kd) {
  constexpr int NWV = 4, NS = KIND >= 0 && KIND < 16 ? 2 : 1, D = MT <= 2 ? 4 : 2, NT = MT * NS;
  using S = OwnRows<MT, NS, D, ONCE>;
  static_assert(NT <= S::BYTES / 1024, "");
  __shared__ __attribute__((aligned(1024))) char smem[NWV * S::BYTES];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int n[NS];
  const bool pair = rows_tiles<KIND>(blockIdx.x, o.f, n);
  const int per = ((Kd + 63) / 64 + NWV - 1) / NWV * 64, k0 = min(wave * per, Kd);  // a wave's k begin at a line
  LineSrc src[NS + MT];
#pragma unroll
  for (int t = 0; t < NS; ++t) src[t] = line_src([&](int r) { return W + (long)min(n[t] + r, o.N - 1) * Kd + k0; });
#pragma unroll
  for (int m = 0; m < MT; ++m) src[NS + m] = line_src([&](int r) { return X + (long)min(16 * m + r, o.M - 1) * x_stride + k0; });
  f32x4 acc[MT][NS] = {};
  S::run(smem + wave * S::BYTES, src, min(per, Kd - k0), acc);
  __syncthreads();  // the rings have been read
  f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NS; ++t) red[(wave * NT + m * NS + t) * 64 + lane] = acc[m][t];
  __syncthreads();
  // element i of lane l: row 4 (l / 16) + i, column l % 16
  auto sum = [&](int m, int t, int l) {
    f32x4 v = red[(m * NS + t) * 64 + l];
#pragma unroll
    for (int g = 1; g < NWV; ++g) v += red[(g * NT + m * NS + t) * 64 + l];
    return v;
  };
  for (int i = threadIdx.x; i < (pair ? MT : NT) * 64; i += 64 * NWV) {
    const int l = i & 63, q = i >> 6, m = pair ? q : q / NS, t = pair ? 0 : q % NS, c = l & 15, r = 16 * m + 4 * (l >> 4);
    const f32x4 v = sum(m, t, l);
    if (pair) {
      const f32x4 u = sum(m, NS - 1, l);
#pragma unroll
      for (int j = 0; j < 4; ++j) rows_store_unit<KIND>(o, r + j, n[0] + c, v[j], u[j]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) rows_store<KIND>(o, r + j, n[NS > 1 ? t : 0] + c, v[j]);
    }
  }
}

template <int KIND, int MT, bool ONCE>
__global__ __launch_bounds__(256) void few_rows_shared_kernel(RowsOut o, const bf16_t* __restrict__ X, long x_stride,
                                                              const bf16_t* __restrict__ W, int Kd) {
  constexpr int NW = 4, NS = KIND >= 0 && KIND < 16 ? 2 : 1;
  using S = SharedRows<MT, NS, NW, ONCE>;
  __shared__ __attribute__((aligned(1024))) char smem[S::BYTES];
  int n[NS];
  const bool pair = rows_tiles<KIND>(blockIdx.x * NW + (threadIdx.x >> 6), o.f, n);
  LineSrc w[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) w[t] = line_src([&](int r) { return W + (long)min(n[t] + r, o.N - 1) * Kd; });
  f32x4 acc[MT][NS] = {};
  S::run(smem, [&](int m) {
    return line_src([&](int r) { return X + (long)min(16 * m + r, o.M - 1) * x_stride; });
  }, w, Kd, acc);
  const int c = threadIdx.x & 15, quad = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * m + 4 * quad + i;
      if (pair) {
        rows_store_unit<KIND>(o, r, n[0] + c, acc[m][0][i], acc[m][NS - 1][i]);
      } else {
#pragma unroll
        for (int t = 0; t < NS; ++t) rows_store<KIND>(o, r, n[t] + c, acc[m][t][i]);
      }
    }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

// kind: see RowsOut (gated: yg [M][f], y [M][N - 2 f]); f32: y is fp32, capped if cap > 0 (kind -1); shared: the form
int k8sllm_hy_few_rows(void* y, void* yg, const void* x, long x_stride, const void* w, int M, int N, int Kd, int f, int kind, int f32,
                       float cap, int shared, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  const bool gated = kind >= 0 && kind < 16;
  if (M > 64 || Kd < 32 || Kd % 32 || x_stride % 8 || (f32 && kind != -1)) return -1;
  if (gated ? f <= 0 || f % 16 || N < 2 * f || yg == nullptr : f != 0) return -1;
  const RowsOut o{y, (bf16_t*)yg, M, N, f, f32, cap};
  const unsigned tiles = (unsigned)(gated ? f / 16 + (N - 2 * f + 31) / 32 : (N + 15) / 16);
  // (shared, 16 rows, 10240 x 384, us, non-temporal / as usual: 15 such weights in turn, which the memory-side cache holds, 5.3 / 4.5; 100 of them, from
  // memory, 5.0 / 5.3; 12288 x 320 4.8 / 4.3, 4.5 / 4.75)
  const bool once = read_once(2l * N * Kd, w, Kd);
#define K8SLLM_FRX(KERNEL, GRID) \
  hipLaunchKernelGGL(KERNEL, dim3(GRID), dim3(256), 0, s, o, (const bf16_t*)x, x_stride, (const bf16_t*)w, Kd)
#define K8SLLM_FR(KIND, MT)                                                                    \
  if (shared && once) K8SLLM_FRX((few_rows_shared_kernel<KIND, MT, true>), (tiles + 3) / 4);   \
  else if (shared) K8SLLM_FRX((few_rows_shared_kernel<KIND, MT, false>), (tiles + 3) / 4);     \
  else if (once) K8SLLM_FRX((few_rows_own_kernel<KIND, MT, true>), tiles);                     \
  else K8SLLM_FRX((few_rows_own_kernel<KIND, MT, false>), tiles)
#define K8SLLM_FRM(KIND)              \
  if (M <= 16) { K8SLLM_FR(KIND, 1); } \
  else if (M <= 32) { K8SLLM_FR(KIND, 2); } \
  else { K8SLLM_FR(KIND, 4); }
  if (kind == -1) { K8SLLM_FRM(-1) }
  else if (kind == 1) { K8SLLM_FRM(1) }
  else if (kind == 3) { K8SLLM_FRM(3) }
  else if (kind == 4) { K8SLLM_FRM(4) }
  else if (kind == 16 + 6) { K8SLLM_FRM(16 + 6) }
  else if (kind == 16 + 7) { K8SLLM_FRM(16 + 7) }
  else return -1;
#undef K8SLLM_FRM
#undef K8SLLM_FR
#undef K8SLLM_FRX
  return (int)hipGetLastError();
}
}
