// Y[M][N] = X[M][K] W[N][K]^T for the few rows of a decode step (bf16, fp32 sums, M up to 16, K a multiple of 32).
// A projection of one or a few rows is a pass over its weights: at the widths of a small model that is 1 to 3 us of memory traffic,
// and what a call takes is set by how soon enough loads are in flight.  A workgroup takes 16 output columns and its 16 waves a
// slice of K each, both operands as 16-byte fragments of v_mfma_f32_16x16x32_bf16 straight from global memory, a batch of loads
// in flight while the last is multiplied; the waves' sums meet in LDS in the order of K.
// us, the BLAS library's call against this one, 1 and 16 rows (N x K): 1024 x 1024 5.6 / 4.1, 5.7 / 5.4; 4096 x 1024 7.5 / 4.7, 7.6 /
// 6.0; 1024 x 4096 14.4 / 7.1, 14.5 / 9.6; 2048 x 2048 11.0 / 4.8, 11.2 / 6.3; 4096 x 4096 15.5 / 9.3, 15.6 / 10.7.  Eight waves:
// up to 0.9 more.  Past the caller's limits the library is faster: 2048 x 5632 10.3 / 10.3, 11.2 / 15.2 (too few workgroups);
// 32000 x 1024 18.7 / 25.5; 16384 x 4096 at 16 rows 33.4 / 39.0.
#include "hy_common.h"

namespace k8sllm {

constexpr int NWV = 16;

// KIND >= 0: W's first 2 f rows are a gated unit's gate and up rows, Yg [M][f] = act(gate) * up of the products rounded to bf16 (as
// the separate launch finds them), each workgroup below f / 16 taking 16 columns of both; Y gets the products of the rest.  One launch less a gated
// feed-forward: a step with six of them (one row, width 1024, f 2816) 422 -> 404 us.
template <int KIND>
__global__ __launch_bounds__(64 * NWV) void few_rows_kernel(bf16_t* __restrict__ Y, const bf16_t* __restrict__ X, long x_stride,
                                                             const bf16_t* __restrict__ W, int M, int N, int Kd,
                                                             bf16_t* __restrict__ Yg, int f) {
  constexpr int U = 4;
  constexpr bool GLU = KIND >= 0;
  __shared__ __attribute__((aligned(16))) float red[GLU ? 2 : 1][NWV][64][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, quad = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const bool pair = GLU && n0 < f;  // uniform
  const int m0 = GLU && !pair ? n0 + f : n0;  // first row of W
  const int per = (Kd / 32 + NWV - 1) / NWV, s0 = min(wave * per, Kd / 32), ns = min(per, Kd / 32 - s0);
  const bf16_t* wp = W + (long)min(m0 + c16, N - 1) * Kd + 32 * s0 + 8 * quad;
  const bf16_t* up = wp + (pair ? (long)f * Kd : 0);
  const bf16_t* xp = X + (long)min(c16, M - 1) * x_stride + 32 * s0 + 8 * quad;
  f32x4 acc = {}, accu = {};
  bf16x8 a[2][U], w[2][U], u[2][U];
  auto load = [&](int h, int i, int k) {
    w[h][i] = *reinterpret_cast<const bf16x8*>(wp + 32 * k);
    if (GLU) u[h][i] = *reinterpret_cast<const bf16x8*>(up + 32 * k);
    a[h][i] = *reinterpret_cast<const bf16x8*>(xp + 32 * k);
  };
  const int nb = (ns + U - 1) / U;  // the last batch repeats its last step's loads and leaves their products out
  if (ns > 0)
#pragma unroll
    for (int i = 0; i < U; ++i) load(0, i, min(i, ns - 1));
  for (int k = 0; k < nb; k += 2) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (k + h >= nb) break;
      if (k + h + 1 < nb)
#pragma unroll
        for (int i = 0; i < U; ++i) load(h ^ 1, i, min((k + h + 1) * U + i, ns - 1));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < U; ++i)
        if ((k + h) * U + i < ns) {
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][i], w[h][i], acc, 0, 0, 0);
          if (GLU) accu = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][i], u[h][i], accu, 0, 0, 0);
        }
    }
  }
  *reinterpret_cast<f32x4*>(red[0][wave][lane]) = acc;
  if (GLU) *reinterpret_cast<f32x4*>(red[GLU][wave][lane]) = accu;
  __syncthreads();
  if (threadIdx.x < 256) {  // element i of lane l: row 4 (l / 16) + i, column l % 16
    const int r = threadIdx.x >> 4, l = (r >> 2) * 16 + c16, i = r & 3;
    if (r >= M || m0 + c16 >= N) return;
    float v = red[0][0][l][i];
#pragma unroll
    for (int g = 1; g < NWV; ++g) v += red[0][g][l][i];
    if (pair) {
      float t = red[GLU][0][l][i];
#pragma unroll
      for (int g = 1; g < NWV; ++g) t += red[GLU][g][l][i];
      Yg[(long)r * f + n0 + c16] = f2bf(glu_unit<GLU ? KIND : 3>(bf2f(f2bf(v)), bf2f(f2bf(t)), 0.f));
    } else {
      const int o = GLU ? 2 * f : 0;
      Y[(long)r * (N - o) + m0 + c16 - o] = f2bf(v);
    }
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

int k8sllm_hy_few_rows(void* y, const void* x, long x_stride, const void* w, int M, int N, int Kd, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || Kd < 32 || Kd % 32 || x_stride % 8) return -1;
  hipLaunchKernelGGL((few_rows_kernel<-1>), dim3((unsigned)((N + 15) / 16)), dim3(64 * NWV), 0, s, (bf16_t*)y, (const bf16_t*)x, x_stride,
                     (const bf16_t*)w, M, N, Kd, (bf16_t*)nullptr, 0);
  return (int)hipGetLastError();
}

// yg [M][f]: the gated unit (kind 1 tanh GELU, 3 SiLU, 4 ReLU) of w's first 2 f rows; y [M][N - 2 f]: the other rows' products
int k8sllm_hy_few_rows_glu(void* yg, void* y, const void* x, long x_stride, const void* w, int M, int N, int Kd, int f, int kind,
                           hipStream_t s) {
  if (M <= 0 || f <= 0) return 0;
  if (M > 16 || Kd < 32 || Kd % 32 || x_stride % 8 || f % 16 || N < 2 * f) return -1;
  const dim3 grid((unsigned)(f / 16 + (N - 2 * f + 15) / 16));
#define K8SLLM_FRG(K)                                                                                                   \
  hipLaunchKernelGGL((few_rows_kernel<K>), grid, dim3(64 * NWV), 0, s, (bf16_t*)y, (const bf16_t*)x, x_stride, (const bf16_t*)w, M, N, \
                     Kd, (bf16_t*)yg, f)
  if (kind == 1) K8SLLM_FRG(1);
  else if (kind == 3) K8SLLM_FRG(3);
  else if (kind == 4) K8SLLM_FRG(4);
  else return -1;
#undef K8SLLM_FRG
  return (int)hipGetLastError();
}
}
