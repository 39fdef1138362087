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

__global__ __launch_bounds__(64 * NWV) void few_rows_kernel(bf16_t* __restrict__ Y, const bf16_t* __restrict__ X, long x_stride,
                                                                   const bf16_t* __restrict__ W, int M, int N, int Kd) {
  constexpr int U = 4;
  __shared__ __attribute__((aligned(16))) float red[NWV][64][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c16 = lane & 15, quad = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int per = (Kd / 32 + NWV - 1) / NWV, s0 = min(wave * per, Kd / 32), ns = min(per, Kd / 32 - s0);
  const bf16_t* wp = W + (long)min(n0 + c16, N - 1) * Kd + 32 * s0 + 8 * quad;
  const bf16_t* xp = X + (long)min(c16, M - 1) * x_stride + 32 * s0 + 8 * quad;
  f32x4 acc = {};
  bf16x8 a[2][U], w[2][U];
  auto load = [&](bf16x8& x, bf16x8& v, int k) {
    v = *reinterpret_cast<const bf16x8*>(wp + 32 * k);
    x = *reinterpret_cast<const bf16x8*>(xp + 32 * k);
  };
  const int nb = (ns + U - 1) / U;  // the last batch repeats its last step's loads and leaves their products out
  if (ns > 0)
#pragma unroll
    for (int i = 0; i < U; ++i) load(a[0][i], w[0][i], min(i, ns - 1));
  for (int k = 0; k < nb; k += 2) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (k + h >= nb) break;
      if (k + h + 1 < nb)
#pragma unroll
        for (int i = 0; i < U; ++i) load(a[h ^ 1][i], w[h ^ 1][i], min((k + h + 1) * U + i, ns - 1));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < U; ++i)
        if ((k + h) * U + i < ns) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[h][i], w[h][i], acc, 0, 0, 0);
    }
  }
  *reinterpret_cast<f32x4*>(red[wave][lane]) = acc;
  __syncthreads();
  if (threadIdx.x < 256) {  // element i of lane l: row 4 (l / 16) + i, column n0 + l % 16
    const int r = threadIdx.x >> 4, l = (r >> 2) * 16 + c16, i = r & 3, n = n0 + c16;
    if (r >= M || n >= N) return;
    float v = red[0][l][i];
#pragma unroll
    for (int g = 1; g < NWV; ++g) v += red[g][l][i];
    Y[(long)r * N + n] = f2bf(v);
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

int k8sllm_hy_few_rows(void* y, const void* x, long x_stride, const void* w, int M, int N, int Kd, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || Kd < 32 || Kd % 32 || x_stride % 8) return -1;
  const dim3 grid((unsigned)((N + 15) / 16));
  hipLaunchKernelGGL(few_rows_kernel, grid, dim3(64 * NWV), 0, s, (bf16_t*)y, (const bf16_t*)x, x_stride, (const bf16_t*)w, M, N, Kd);
  return (int)hipGetLastError();
}
}
