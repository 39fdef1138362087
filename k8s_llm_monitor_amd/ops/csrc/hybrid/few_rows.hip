// Y[M][N] = X[M][K] W[N][K]^T for the few rows of a decode step (bf16, fp32 sums, M up to 64, K a multiple of 32).
// A projection of a few rows is a pass over its weights; what a call takes is set by how soon enough loads are in flight, and by how
// often the rows are fetched beside the weights.  Two forms (stream_rows.h has the streams):
//   own     a workgroup takes 16 columns, its four waves a quarter of K each with their own copies of the rows; the waves' sums meet in
//           LDS in the order of K.  As many workgroups as there are column tiles.
//   shared  a workgroup takes 64 columns and all of K, its four waves share the rows.
#include "split_bf16.h"
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

// ONCE, TURN: the weights non-temporal, and from a k of the workgroup's own on (a kernel of its own: the address of a line that is not
// turned costs a small product 0.15 us otherwise)
template <int KIND, int MT, bool ONCE, bool TURN = false>
__global__ __launch_bounds__(256) void few_rows_own_kernel(RowsOut o, const bf16_t* __restrict__ X, long x_stride,
                                                           const bf16_t* __restrict__ W, int Kd) {
  constexpr int NWV = 4, NS = KIND >= 0 && KIND < 16 ? 2 : 1, D = MT <= 2 ? 4 : 2, NT = MT * NS;
  using S = OwnRows<MT, NS, D, ONCE, TURN>;
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
  S::run(smem + wave * S::BYTES, src, min(per, Kd - k0), acc, TURN ? 4 * first_piece(blockIdx.x, per / 256) : 0);
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

template <int KIND, int MT, bool ONCE, bool TURN = false>
__global__ __launch_bounds__(256) void few_rows_shared_kernel(RowsOut o, const bf16_t* __restrict__ X, long x_stride,
                                                              const bf16_t* __restrict__ W, int Kd) {
  constexpr int NW = 4, NS = KIND >= 0 && KIND < 16 ? 2 : 1;
  using S = SharedRows<MT, NS, NW, ONCE, TURN>;
  __shared__ __attribute__((aligned(1024))) char smem[S::BYTES];
  int n[NS];
  const bool pair = rows_tiles<KIND>(blockIdx.x * NW + (threadIdx.x >> 6), o.f, n);
  LineSrc w[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) w[t] = line_src([&](int r) { return W + (long)min(n[t] + r, o.N - 1) * Kd; });
  f32x4 acc[MT][NS] = {};
  S::run(smem, [&](int m) {
    return line_src([&](int r) { return X + (long)min(16 * m + r, o.M - 1) * x_stride; });
  }, w, Kd, acc, TURN ? first_piece(blockIdx.x, Kd / 256) : 0);
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

// Rows that are made here: the gated residual's sum and its norm (gated_add_norm_kernel, the same sums in the same order) are every workgroup's
// prologue, behind the first loads of its weights, so the norm is no launch of its own.  Workgroup 0 writes the new residual, to a buffer of its own
// (the others still read the old one).  What it costs is one round of loads, some 200 instructions a row and two barriers in each workgroup, against a
// launch: few rows only.  us, norm and product / this, weights from memory: 1 row 3584 x 1024 5.9 / 4.4, 7168 x 2048 9.3 / 7.4, gated unit of 5632 + 2048
// columns x 2048 15.3 / 11.3; 2 rows 3584 x 1024 5.9 / 4.6, 7168 x 2048 9.2 / 8.8; 4 rows 3584 x 1024 6.2 / 5.6, unit of 2816 + 1024 7.8 / 7.5, 7168 x
// 2048 9.8 / 11.5; 1 row of 4096 columns 14336 x 4096 24.3 / 29.8.
struct GatedRows {
  const float* x;  // [M][Kd], and the new one
  float* xn;
  const bf16_t *y, *gate;  // [M][Kd]; rows g_stride apart
  long g_stride;
  const float *bias, *w;
  float mult, eps;
  int one_plus;
};

// KIND as above.  M <= MR rows of Kd <= 2048 / RP columns: RP rows at a time, each by 4 / RP waves.  As few_rows_own_kernel: 16 columns a workgroup,
// its waves a quarter of K each.
template <int KIND, int MR, int RP, bool ONCE>
__global__ __launch_bounds__(256) void few_rows_gated_kernel(RowsOut o, GatedRows g, const bf16_t* __restrict__ W, int Kd) {
  constexpr int NWV = 4, NS = KIND >= 0 && KIND < 16 ? 2 : 1, D = 4, P = MR / RP, RW = NWV / RP;
  using S = HeldRows<NS, D, ONCE>;
  __shared__ __attribute__((aligned(1024))) char smem[NWV * S::BYTES];
  __shared__ __attribute__((aligned(16))) bf16_t xs[MR * (2048 / RP + 32)];
  __shared__ float red[MR][RW];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), pitch = Kd + 32;
  const int half = wave / RW, at = 8 * (threadIdx.x - 64 * RW * half), c = min(at, Kd - 8);  // a thread past the row's end adds nothing
  float x[P][8], b[8], nw[8];
  uint4 y[P], gt[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const long row = min(RP * p + half, o.M - 1);
    load8(g.x + row * Kd + c, x[p]);
    y[p] = *reinterpret_cast<const uint4*>(g.y + row * Kd + c);
    gt[p] = *reinterpret_cast<const uint4*>(g.gate + row * g.g_stride + c);
  }
  load8(g.bias + c, b);
  load8(g.w + c, nw);
  int n[NS];
  const bool pair = rows_tiles<KIND>(blockIdx.x, o.f, n);
  const int per = ((Kd + 63) / 64 + NWV - 1) / NWV * 64, k0 = min(wave * per, Kd);  // a wave's k begin at a line
  const int kd = min(per, Kd - k0);
  LineSrc w[NS];
#pragma unroll
  for (int t = 0; t < NS; ++t) w[t] = line_src([&](int r) { return W + (long)min(n[t] + r, o.N - 1) * Kd + k0; });
  char* ring = smem + wave * S::BYTES;
  S::begin(ring, w, kd);
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int r = RP * p + half;
    float ss = 0.f, a[8], z[8];
    unpack8(y[p], a);
    unpack8(gt[p], z);
    if (at < Kd) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        x[p][i] += g.mult * a[i] * sigmoid_f(z[i] + b[i]);
        ss += x[p][i] * x[p][i];
      }
      if (blockIdx.x == 0 && r < o.M) store8(g.xn + (long)r * Kd + c, x[p]);
    }
    ss = wave_sum(ss);
    if (lane == 0) red[r][wave - RW * half] = ss;
  }
  lds_barrier();
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const int r = RP * p + half;
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < RW; ++i) t += red[r][i];
    const float inv = 1.0f / sqrtf(t / (float)Kd + g.eps);
    if (at < Kd) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[p][i] *= inv * (g.one_plus ? 1.f + nw[i] : nw[i]);
      *reinterpret_cast<uint4*>(xs + r * pitch + c) = pack8(x[p]);
    }
  }
  lds_barrier();
  f32x4 acc[NS] = {};
  S::run(ring, w, xs + min(lane & 15, MR - 1) * pitch + k0 + 8 * (lane >> 4), kd, acc);
  __syncthreads();  // the rings have been read
  f32x4* sums = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int t = 0; t < NS; ++t) sums[(wave * NS + t) * 64 + lane] = acc[t];
  __syncthreads();
  // element i of lane l: row 4 (l / 16) + i, column l % 16: the rows are lanes 0 to 15's
  const int l = threadIdx.x & 15, t = threadIdx.x >> 4;
  if (t >= (pair ? 1 : NS)) return;
  auto sum = [&](int q) {
    f32x4 v = sums[q * 64 + l];
#pragma unroll
    for (int k = 1; k < NWV; ++k) v += sums[(k * NS + q) * 64 + l];
    return v;
  };
  const f32x4 v = sum(t);
  if (pair) {
    const f32x4 u = sum(NS - 1);
#pragma unroll
    for (int j = 0; j < MR; ++j) rows_store_unit<KIND>(o, j, n[0] + l, v[j], u[j]);
  } else {
#pragma unroll
    for (int j = 0; j < MR; ++j) rows_store<KIND>(o, j, n[NS > 1 ? t : 0] + l, v[j]);
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
  // workgroups begin at k of their own (first_piece) where a wave's rows, or its quarters of them, are whole periods of the channels, and there are
  // enough of them to meet in one
  const bool turn = once && (shared ? (tiles + 3) / 4 : tiles) >= kTurnGroups && Kd % (shared ? kTurnBytes / 2 : 2 * kTurnBytes) == 0;
#define K8SLLM_FRX(KERNEL, GRID) \
  hipLaunchKernelGGL(KERNEL, dim3(GRID), dim3(256), 0, s, o, (const bf16_t*)x, x_stride, (const bf16_t*)w, Kd)
#define K8SLLM_FR(KIND, MT)                                                                                \
  if (shared && turn) K8SLLM_FRX((few_rows_shared_kernel<KIND, MT, true, true>), (tiles + 3) / 4);         \
  else if (shared && once) K8SLLM_FRX((few_rows_shared_kernel<KIND, MT, true>), (tiles + 3) / 4);          \
  else if (shared) K8SLLM_FRX((few_rows_shared_kernel<KIND, MT, false>), (tiles + 3) / 4);                 \
  else if (turn) K8SLLM_FRX((few_rows_own_kernel<KIND, MT, true, true>), tiles);                           \
  else if (once) K8SLLM_FRX((few_rows_own_kernel<KIND, MT, true>), tiles);                                 \
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

// The same of rows made in the prologue (see GatedRows): x, y, xn [M][Kd] contiguous, 16-byte aligned, as are gate's rows, bias and w.
int k8sllm_hy_few_rows_gated(void* y, void* yg, const float* x, float* xn, const void* add, const void* gate, long g_stride,
                             const float* bias, float mult, const float* nw, float eps, int one_plus, const void* w, int M, int N, int Kd,
                             int f, int kind, hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  const bool gated = kind >= 0;
  if (M > 4 || Kd > (M > 2 ? 1024 : 2048) || Kd < 32 || Kd % 32 || g_stride % 8) return -1;
  if (gated ? f <= 0 || f % 16 || N < 2 * f || yg == nullptr : f != 0) return -1;
  const RowsOut o{y, (bf16_t*)yg, M, N, f, 0, 0.f};
  const GatedRows g{x, xn, (const bf16_t*)add, (const bf16_t*)gate, g_stride, bias, nw, mult, eps, one_plus};
  const unsigned tiles = (unsigned)(gated ? f / 16 + (N - 2 * f + 31) / 32 : (N + 15) / 16);
  const bool once = read_once(2l * N * Kd, w, Kd);
#define K8SLLM_FGX(KIND, MR, RP, ONCE) \
  hipLaunchKernelGGL((few_rows_gated_kernel<KIND, MR, RP, ONCE>), dim3(tiles), dim3(256), 0, s, o, g, (const bf16_t*)w, Kd)
#define K8SLLM_FGO(KIND, MR, RP)                 \
  if (once) { K8SLLM_FGX(KIND, MR, RP, true); } \
  else { K8SLLM_FGX(KIND, MR, RP, false); }
#define K8SLLM_FG(KIND)                                   \
  if (M == 1) { K8SLLM_FGO(KIND, 1, 1) }                  \
  else if (Kd > 1024) { K8SLLM_FGO(KIND, 2, 1) }          \
  else if (M == 2) { K8SLLM_FGO(KIND, 2, 2) }             \
  else { K8SLLM_FGO(KIND, 4, 2) }
  if (kind == -1) { K8SLLM_FG(-1) }
  else if (kind == 1) { K8SLLM_FG(1) }
  else if (kind == 3) { K8SLLM_FG(3) }
  else if (kind == 4) { K8SLLM_FG(4) }
  else return -1;
#undef K8SLLM_FG
#undef K8SLLM_FGO
#undef K8SLLM_FGX
  return (int)hipGetLastError();
}
}
