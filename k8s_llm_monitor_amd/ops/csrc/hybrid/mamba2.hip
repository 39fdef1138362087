// Mamba-2 mixer kernels (any sizes; state and recurrence fp32).
//   conv_silu        causal per-channel convolution (bias optional) + SiLU over a column range of the in-projection,
//                    one thread per (row, channel); the taps-1 inputs before a segment come from the
//                    sequence's conv state slot (zeros for a sequence that starts in this step)
//   conv_state_step  advances each segment's conv state slot to the segment's end
//   ssm_scan         S <- exp(-exp(A_log) dt) S + dt B x^T;  y = S^T C + D x, token by token per
//                    segment; the state slot [nh][N][P] is read at the start, written at the end.
//                    With a table of fixed decays per head (``decay``) the same scan is the linear
//                    attention recurrence S <- decay S + k v^T, y = S^T q (dt = 1, no skip term; B, C, x
//                    are k, q, v)
// A segment is one sequence's rows of this step: cu[s] .. cu[s+1], ctx[s] tokens already in its
// state (0: starts from zero), slot[s] its state slot (< 0: skipped).
#include "hy_common.h"

namespace k8sllm {

constexpr int kMaxTaps = 16;

// Sum over groups of CH consecutive lanes (CH a power of two <= 32, groups aligned); lane 0 of each
// group holds the group's total afterwards (every lane of the group does, up to CH = 16).  Row-local
// DPP adds (one VALU instruction each, no LDS crossbar): quads by quad_perm, then the row's halves
// and the row by the mirror controls, which pair equal partial sums.
template <int CH>
__device__ __forceinline__ float group_sum(float v) {
  if (CH >= 2) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));
  if (CH >= 4) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true));
  if (CH >= 8) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, true));
  if (CH >= 16) v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xf, 0xf, true));
  if (CH >= 32) v = xor16_sum(v);
  return v;
}

template <typename T>
__global__ __launch_bounds__(256) void conv_silu_kernel(T* __restrict__ out, const T* __restrict__ proj, long stride,
                                                        int col0, int C, const float* __restrict__ cw,
                                                        const float* __restrict__ cb, int taps,
                                                        const T* __restrict__ state, const int* __restrict__ cu,
                                                        const int* __restrict__ ctx, const int* __restrict__ slot,
                                                        int S) {
  const int row = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= C) return;
  const int s = find_segment(cu, S, row);
  const int sl = slot[s];
  if (sl < 0) {  // padding row: defined output, no state
    stf(out + (long)row * C + c, 0.f);
    return;
  }
  const int r = row - cu[s];
  const bool carried = ctx[s] > 0;
  float acc = cb != nullptr ? cb[c] : 0.f;
  for (int j = 0; j < taps; ++j) {
    const int i = r - (taps - 1) + j;  // offset within the segment of the input under tap j
    float x = 0.f;
    if (i >= 0)
      x = ldf(proj + (long)(row - (taps - 1) + j) * stride + col0 + c);
    else if (carried)
      x = ldf(state + ((long)sl * (taps - 1) + (taps - 1 + i)) * C + c);
    acc += cw[(long)c * taps + j] * x;
  }
  stf(out + (long)row * C + c, silu_f(acc));
}

template <typename T>
struct Raw8 {  // eight values as they lie in memory
  uint4 q[sizeof(T) / 2];
  __device__ __forceinline__ void from(const T* p) {  // 16-byte aligned
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 2); ++i) q[i] = reinterpret_cast<const uint4*>(p)[i];
  }
  __device__ __forceinline__ void from(const T* p, int n, int last) {  // p[n .. n + 7], past `last` that one
    T v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = p[min(n + k, last)];
    __builtin_memcpy(q, v, sizeof(v));
  }
  __device__ __forceinline__ void to(float* f) const { load8(reinterpret_cast<const T*>(q), f); }
};

// The same with 8 channels and R rows per thread (16 / 32-byte accesses): channel count, column offset and row strides multiples
// of 8.  A row's weights are 128 bytes to its 16 of input at the usual 4 taps, so a thread that takes one row (R = 1: the few rows of
// a decode step) mostly reads weights; R rows share them, and inside a segment each row's input is read once for its four taps,
// all of them in flight together.  8000 rows of 4096 channels bf16: 89 -> 38 us, 3.5 TB/s.
template <typename T, int R>
__global__ __launch_bounds__(256) void conv_silu_vec8_kernel(T* __restrict__ out, const T* __restrict__ proj,
                                                             long stride, int col0, int C, const float* __restrict__ cw,
                                                             const float* __restrict__ cb, int taps,
                                                             const T* __restrict__ state, const int* __restrict__ cu,
                                                             const int* __restrict__ ctx, const int* __restrict__ slot,
                                                             int S, int rows) {
  const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (c >= C) return;
  const int row0 = blockIdx.x * R;
  float4 wv[8];
  if (taps == 4) {
#pragma unroll
    for (int k = 0; k < 8; ++k) wv[k] = *reinterpret_cast<const float4*>(cw + (long)(c + k) * 4);
  }
  float bias[8];
  if (cb != nullptr) {
    load8(cb + c, bias);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) bias[i] = 0.f;
  }
  int s = find_segment(cu, S, row0);
  if (R > 1 && taps == 4 && row0 + R <= cu[s + 1] && row0 - 3 >= cu[s] && slot[s] >= 0) {  // all inputs lie in one segment
    Raw8<T> in[R + 3];
    const T* px = proj + (long)(row0 - 3) * stride + col0 + c;
#pragma unroll
    for (int i = 0; i < R + 3; ++i) in[i].from(px + i * stride);
    float x[4][8];
#pragma unroll
    for (int i = 0; i < 3; ++i) in[i].to(x[i]);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      in[r + 3].to(x[(r + 3) & 3]);
      float acc[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float v = bias[k];
        v += wv[k].x * x[r & 3][k];
        v += wv[k].y * x[(r + 1) & 3][k];
        v += wv[k].z * x[(r + 2) & 3][k];
        v += wv[k].w * x[(r + 3) & 3][k];
        acc[k] = silu_f(v);
      }
      store8(out + (long)(row0 + r) * C + c, acc);
    }
    return;
  }
  for (int row = row0; row < min(row0 + R, rows); ++row) {
    if (R > 1)
      while (s < S - 1 && row >= cu[s + 1]) ++s;
    const int sl = slot[s];
    float acc[8], x[8];
    if (sl < 0) {  // padding row: defined output, no state
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = 0.f;
      store8(out + (long)row * C + c, acc);
      continue;
    }
    const int r = row - cu[s];
    const bool carried = ctx[s] > 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = bias[i];
    if (taps == 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = r - 3 + j;
        if (i >= 0)
          load8(proj + (long)(row - 3 + j) * stride + col0 + c, x);
        else if (carried)
          load8(state + ((long)sl * 3 + (3 + i)) * C + c, x);
        else
          continue;
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] += (j == 0 ? wv[k].x : j == 1 ? wv[k].y : j == 2 ? wv[k].z : wv[k].w) * x[k];
      }
    } else {
      for (int j = 0; j < taps; ++j) {
        const int i = r - (taps - 1) + j;
        if (i >= 0)
          load8(proj + (long)(row - (taps - 1) + j) * stride + col0 + c, x);
        else if (carried)
          load8(state + ((long)sl * (taps - 1) + (taps - 1 + i)) * C + c, x);
        else
          continue;
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] += cw[(long)(c + k) * taps + j] * x[k];
      }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = silu_f(acc[k]);
    store8(out + (long)row * C + c, acc);
  }
}

// Steps of one token a segment (decode), four taps: eight channels of a segment a thread, which has the history in registers for the output and
// for the slot's new history, so one launch instead of conv_silu_vec8_kernel and conv_state_step_kernel (each read weights or inputs of 2
// bytes behind a search for the row's segment).  The same sums.  us, both / this: 24 sequences of 8192 channels 9.0 / 6.1,
// 64 of 4352 10.7 / 4.7, one of 2048 7.4 / 5.4.
template <typename T>
__global__ __launch_bounds__(256) void conv_step_kernel(T* __restrict__ out, const T* __restrict__ proj, long stride, int col0, int C,
                                                        const float* __restrict__ cw, const float* __restrict__ cb, T* __restrict__ state,
                                                        const int* __restrict__ cu, const int* __restrict__ ctx,
                                                        const int* __restrict__ slot) {
  const int s = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (c >= C) return;
  const int sl = slot[s], t0 = cu[s], t1 = cu[s + 1];
  if (sl < 0) {  // padding rows: defined output, no state
    const float zero[8] = {};
    for (int t = t0; t < t1; ++t) store8(out + (long)t * C + c, zero);
    return;
  }
  if (t1 <= t0) return;
  T* st = state + (long)sl * 3 * C + c;
  Raw8<T> in[4];  // the last four inputs, oldest first
#pragma unroll
  for (int j = 0; j < 3; ++j) in[j].from(st + (long)j * C);
  int have = ctx[s] > 0 ? 3 : 0;  // so many of them before this token's
  float4 wv[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) wv[k] = *reinterpret_cast<const float4*>(cw + (long)(c + k) * 4);
  float bias[8] = {};
  if (cb != nullptr) load8(cb + c, bias);
  for (int t = t0; t < t1; ++t) {
    in[3].from(proj + (long)t * stride + col0 + c);
    float acc[8], x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = bias[k];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      in[j].to(x);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float a = acc[k] + (j == 0 ? wv[k].x : j == 1 ? wv[k].y : j == 2 ? wv[k].z : wv[k].w) * x[k];
        acc[k] = j + have >= 3 ? a : acc[k];
      }
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = silu_f(acc[k]);
    store8(out + (long)t * C + c, acc);
#pragma unroll
    for (int j = 0; j < 3; ++j) in[j] = in[j + 1];
    have = min(have + 1, 3);
  }
  const float zero[8] = {};
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    if (j + have < 3) {
      store8(st + (long)j * C, zero);
    } else {
      float x[8];
      in[j].to(x);
      store8(st + (long)j * C, x);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void conv_state_step_kernel(T* __restrict__ state, const T* __restrict__ proj,
                                                              long stride, int col0, int C, int taps,
                                                              const int* __restrict__ cu, const int* __restrict__ ctx,
                                                              const int* __restrict__ slot) {
  const int s = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  const int sl = slot[s];
  const int n = cu[s + 1] - cu[s];
  if (c >= C || sl < 0 || n <= 0) return;
  const int H = taps - 1;
  const bool carried = ctx[s] > 0;
  T* st = state + (long)sl * H * C + c;
  T keep[kMaxTaps];
  for (int i = 0; i < H; ++i) {  // entry i of the new history = element n + i of [old history ; segment]
    const int k = n + i;
    if (k >= H)
      keep[i] = proj[(long)(cu[s] + k - H) * stride + col0 + c];
    else if (carried)
      keep[i] = st[(long)k * C];
    else
      stf(&keep[i], 0.f);
  }
  for (int i = 0; i < H; ++i) st[(long)i * C] = keep[i];
}

// State 4 i + j behind a token.  Which of the two products is rounded before they meet is the choice that a compiler once made, spelled out:
// a decode step's bits decide near ties of routers behind it.
template <int NPT>
__device__ __forceinline__ float next_state(int j, float dA, float S, float dtx, float b) {
  return NPT == 4 || (NPT < 64 && j == 0) ? fmaf(dA, S, dtx * b) : fmaf(dtx, b, dA * S);
}

// Workgroup = 4 waves = 64 values of p for one (segment, head); in a wave lanes are (p % 16,
// chunk = lane / 16): chunk k holds states n in [k * NPT, (k + 1) * NPT) of its p in registers, and
// the 4 partial sums of y meet through two xor-shuffles.  The inputs of 16 tokens at a time (B, C
// widened to fp32, x, and dt / the decay after softplus and exp) are staged in LDS by the whole
// workgroup, so the token loop reads only LDS (16-byte reads; the chunks' rows are padded apart by
// 4 floats so the 4 chunks of a wave hit different banks) and global latency is paid once per 16
// tokens instead of once per token.
template <typename T, int NPT>
__global__ __launch_bounds__(256) void ssm_scan_kernel(float* __restrict__ y, const T* __restrict__ xbc,
                                                       const T* __restrict__ proj, long p_stride, int dt_col,
                                                       const float* __restrict__ dt_bias,
                                                       const float* __restrict__ a_log,
                                                       const float* __restrict__ d_skip,
                                                       const float* __restrict__ decay, float* __restrict__ state,
                                                       const int* __restrict__ cu, const int* __restrict__ ctx,
                                                       const int* __restrict__ slot, int nh, int P, int N, int G) {
  constexpr int TB = 16;
  constexpr int CS = NPT + 4;
  __shared__ __attribute__((aligned(16))) float Bs[TB][4 * CS];
  __shared__ __attribute__((aligned(16))) float Cs[TB][4 * CS];
  __shared__ float xs[TB][64];
  __shared__ float dts[TB], dAs[TB];
  const int s = blockIdx.x, h = blockIdx.y;
  const int sl = slot[s];
  const int t0 = cu[s], t1 = cu[s + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int pl = wave * 16 + (lane & 15);
  const int p = blockIdx.z * 64 + pl;
  if (sl < 0) {  // padding rows: defined output, no state
    if (p < P && lane < 16)
      for (int t = t0; t < t1; ++t) y[(long)t * nh * P + (long)h * P + p] = 0.f;
    return;
  }
  if (t1 <= t0) return;
  const int chunk = lane >> 4, n0 = chunk * NPT;
  const bool live = p < P;
  const int g = h / (nh / G);
  const int inner = nh * P, C = inner + 2 * G * N;
  for (int i = threadIdx.x; i < TB * 4 * CS; i += 256) {  // entries beyond N stay zero
    (&Bs[0][0])[i] = 0.f;
    (&Cs[0][0])[i] = 0.f;
  }
  float S[NPT];
  float* sp = state + (((long)sl * nh + h) * N) * P + p;
  const bool carried = ctx[s] > 0;
#pragma unroll
  for (int i = 0; i < NPT; ++i) S[i] = (carried && live && n0 + i < N) ? sp[(long)(n0 + i) * P] : 0.f;
  const bool fixed = decay != nullptr;  // fixed decay per head: dt = 1, no skip term
  const float A = fixed ? 0.f : expf(a_log[h]), Dh = fixed ? 0.f : d_skip[h], bias = fixed ? 0.f : dt_bias[h];
  const float dfix = fixed ? decay[h] : 0.f;
  for (int tb = t0; tb < t1; tb += TB) {
    const int nt = min(TB, t1 - tb);
    __syncthreads();  // the previous tile is consumed (and the zero fill is done)
#pragma unroll 8
    for (int i = threadIdx.x; i < nt * N; i += 256) {  // unrolled: the independent loads go out together
      const int tt = i / N, n = i - tt * N;
      const T* row = xbc + (long)(tb + tt) * C + inner + (long)g * N + n;
      const int off = (n / NPT) * CS + n % NPT;
      Bs[tt][off] = ldf(row);
      Cs[tt][off] = ldf(row + (long)G * N);
    }
#pragma unroll 4
    for (int i = threadIdx.x; i < nt * 64; i += 256) {
      const int tt = i >> 6, pp = i & 63;
      const int pg = blockIdx.z * 64 + pp;
      xs[tt][pp] = pg < P ? ldf(xbc + (long)(tb + tt) * C + (long)h * P + pg) : 0.f;
    }
    if (threadIdx.x < nt) {
      if (fixed) {
        dts[threadIdx.x] = 1.f;
        dAs[threadIdx.x] = dfix;
      } else {
        const float raw = ldf(proj + (long)(tb + threadIdx.x) * p_stride + dt_col + h) + bias;
        const float dt = raw > 20.f ? raw : log1pf(expf(raw));
        dts[threadIdx.x] = dt;
        dAs[threadIdx.x] = expf(-A * dt);
      }
    }
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      const float dA = dAs[tt], x = xs[tt][pl];
      const float dtx = dts[tt] * x;
      const float4* bp = reinterpret_cast<const float4*>(&Bs[tt][chunk * CS]);
      const float4* cp = reinterpret_cast<const float4*>(&Cs[tt][chunk * CS]);
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < NPT / 4; ++i) {
        const float4 bv = bp[i], cv = cp[i];
        S[4 * i + 0] = next_state<NPT>(0, dA, S[4 * i + 0], dtx, bv.x);
        S[4 * i + 1] = next_state<NPT>(1, dA, S[4 * i + 1], dtx, bv.y);
        S[4 * i + 2] = next_state<NPT>(2, dA, S[4 * i + 2], dtx, bv.z);
        S[4 * i + 3] = next_state<NPT>(3, dA, S[4 * i + 3], dtx, bv.w);
        acc += S[4 * i + 0] * cv.x + S[4 * i + 1] * cv.y + S[4 * i + 2] * cv.z + S[4 * i + 3] * cv.w;
      }
      acc = xor32_sum_f(xor16_sum(acc));
      if (live && lane < 16) y[(long)(tb + tt) * inner + (long)h * P + p] = acc + Dh * x;
    }
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < NPT; ++i)
      if (n0 + i < N) sp[(long)(n0 + i) * P] = S[i];
  }
}

// Steps of one token a segment (decode): a pass over the states.  A workgroup takes 64 values of p of one (segment, head); a thread
// holds four of them for every sixteenth group of four states, so that rows of the state are read and written 256 bytes at a time, and all of its
// loads are on their way before anything waits.  Groups' sums meet in LDS in the order of ssm_scan_kernel: the same bits.  That kernel's 4-byte
// accesses met 64 bytes of a row, behind the staging of tiles of 16 tokens.
// us, ssm_scan_kernel / here: 64 heads of 64 x 128, 1 segment 9.5 / 4.6, 16 22.6 / 14.5, 64 75.7 / 49.0 (5.5 TB/s), 128 129 / 98;
// 16 heads of 128 x 128 with a fixed decay, 1 segment 8.4 / 3.6, 32 19.5 / 14.1; 64 of them 40.2 / 26.8.  States above 8 MB of a step are
// non-temporal: at 34 MB 18.6 / 14.5.  silu: rows of a projection, read through SiLU and rounded as its own launch leaves them (us, both
// launches / this: 8 heads of 128 x 128, 1 sequence 5.4 / 4.2, 64 13.2 / 11.1; 32 heads, 16 sequences 12.7 / 11.0).
template <typename T, int NPT, bool ONCE>
__global__ __launch_bounds__(256) void ssm_step_kernel(float* __restrict__ y, const T* __restrict__ xbc, const T* __restrict__ proj,
                                                       long p_stride, int dt_col, const float* __restrict__ dt_bias,
                                                       const float* __restrict__ a_log, const float* __restrict__ d_skip,
                                                       const float* __restrict__ decay, float* __restrict__ state,
                                                       const int* __restrict__ cu, const int* __restrict__ ctx,
                                                       const int* __restrict__ slot, int nh, int P, int N, int G, long x_stride,
                                                       int silu) {
  constexpr int GPT = NPT <= 16 ? 1 : NPT / 16;  // groups of a thread
  __shared__ __attribute__((aligned(16))) float part[16 * GPT][68];
  const int s = blockIdx.x, h = blockIdx.y, sl = slot[s], t0 = cu[s], t1 = cu[s + 1];
  const int lane = threadIdx.x & 63, tg = threadIdx.x >> 4, p4 = blockIdx.z * 64 + 4 * (threadIdx.x & 15);
  const int chunk = lane >> 4, pl = (threadIdx.x >> 6) * 16 + (lane & 15), p = blockIdx.z * 64 + pl;  // as in ssm_scan_kernel
  if (sl < 0) {  // padding rows: defined output, no state
    if (p < P && lane < 16)
      for (int t = t0; t < t1; ++t) y[(long)t * nh * P + (long)h * P + p] = 0.f;
    return;
  }
  if (t1 <= t0) return;
  const int inner = nh * P, g = h / (nh / G), pc = min(p4, P - 4);
  float* sp = state + ((long)sl * nh + h) * N * P + pc;
  int n[GPT];
#pragma unroll
  for (int i = 0; i < GPT; ++i) n[i] = min(4 * (tg + 16 * i), N - 4);  // groups behind the last repeat it, and nothing reads them
  f32v4 S[GPT][4];
  const bool carried = ctx[s] > 0;
#pragma unroll
  for (int i = 0; i < GPT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) S[i][j] = load_state<ONCE>(sp + (long)(n[i] + j) * P);
  const bool fixed = decay != nullptr;
  const float A = fixed ? 0.f : expf(a_log[h]), Dh = fixed ? 0.f : d_skip[h], bias = fixed ? 0.f : dt_bias[h];
  for (int t = t0; t < t1; ++t) {
    const T* row = xbc + (long)t * x_stride;
    float x[4], b[GPT][4], c[GPT][4];
    load4(row + (long)h * P + pc, x);
#pragma unroll
    for (int i = 0; i < GPT; ++i) {
      load4(row + inner + (long)g * N + n[i], b[i]);
      load4(row + inner + (long)(G + g) * N + n[i], c[i]);
    }
    const float xl = ldf(row + (long)h * P + min(p, P - 1));
    if (silu) {
      auto unit = [](float (&v)[4]) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          T r;
          stf(&r, act_f<3>(v[k], 0.f, 0.f));
          v[k] = ldf(&r);
        }
      };
      unit(x);
#pragma unroll
      for (int i = 0; i < GPT; ++i) {
        unit(b[i]);
        unit(c[i]);
      }
    }
    float dt = 1.f, dA;
    if (fixed) {
      dA = decay[h];
    } else {
      const float raw = ldf(proj + (long)t * p_stride + dt_col + h) + bias;
      dt = raw > 20.f ? raw : log1pf(expf(raw));
      dA = expf(-A * dt);
    }
    if (t == t0 && !carried) {
#pragma unroll
      for (int i = 0; i < GPT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) S[i][j] = f32v4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < GPT; ++i) {
      f32v4 sum;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float dtx = dt * x[v];
#pragma unroll
        for (int j = 0; j < 4; ++j) S[i][j][v] = next_state<NPT>(j, dA, S[i][j][v], dtx, b[i][j]);
        sum[v] = fmaf(S[i][3][v], c[i][3], fmaf(S[i][2][v], c[i][2], fmaf(S[i][0][v], c[i][0], S[i][1][v] * c[i][1])));
      }
      *reinterpret_cast<f32v4*>(&part[tg + 16 * i][4 * (threadIdx.x & 15)]) = sum;
    }
    __syncthreads();
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < NPT / 4; ++i) {
      const int q = chunk * (NPT / 4) + i;
      acc += 4 * q < N ? part[q][pl] : 0.f;
    }
    acc = xor32_sum_f(xor16_sum(acc));
    if (p < P && lane < 16) y[(long)t * inner + (long)h * P + p] = fmaf(Dh, xl, acc);
    if (t + 1 < t1) __syncthreads();
  }
  if (p4 < P) {
#pragma unroll
    for (int i = 0; i < GPT; ++i)
      if (4 * (tg + 16 * i) < N) {
#pragma unroll
        for (int j = 0; j < 4; ++j) store_state<ONCE>(sp + (long)(n[i] + j) * P, S[i][j]);
      }
  }
}

// Long segments (prompts): the same recurrence with the state spread thinner - 8 states per lane, CH = N / 8 lanes per value of p
// (their partial sums meet in DPP adds over neighbouring lanes), 64 / CH values of p per wave.  The token loop is sequential per
// (sequence, head, p), so a prompt's scan takes what a token costs a wave: three VALU instructions per state, the DPP adds and
// the LDS reads of B and C.  Everything else is kept out of that loop: a tile of 16 tokens is fetched into registers (16 bytes a load where `vec` says so) while the one
// before it runs, step sizes and decays are computed for 256 tokens at a time, one per thread, and a tile's read-outs meet in LDS
// (lane k of a group keeps token k's) and leave as rows.  State rows are read and written with a stride here, which is why
// single-token segments (decode) keep the mapping above.
// 4 prompts of 2048 tokens, 64 heads of 64 x 128 bf16: 850 us when every tile waited for its loads and computed its own step
// sizes and every token stored its own read-outs, 625 now, the vector unit busy throughout; the mapping below takes the shapes
// that it can (464).  The products and sums are spelled out: both mappings give the same bits.
template <typename T, int CH>
__global__ __launch_bounds__(256) void ssm_scan_wide_kernel(float* __restrict__ y, const T* __restrict__ xbc,
                                                            const T* __restrict__ proj, long p_stride, int dt_col,
                                                            const float* __restrict__ dt_bias,
                                                            const float* __restrict__ a_log,
                                                            const float* __restrict__ d_skip,
                                                            const float* __restrict__ decay,
                                                            float* __restrict__ state, const int* __restrict__ cu,
                                                            const int* __restrict__ ctx, const int* __restrict__ slot,
                                                            int nh, int P, int N, int G, int vec) {
  constexpr int TB = 16, PW = 64 / CH, PB = 4 * PW, LB = 256;
  constexpr int ROW = 8 * CH + (CH / 8) * 4 + 4;  // state n sits at n + 4 (n / 64): 64-float halves 4 banks apart
  constexpr int GR = CH < TB ? CH : TB;           // tokens whose read-outs the lanes of a group keep
  constexpr int NB = (TB * CH + 255) / 256, NX = (TB * PB + 255) / 256;
  __shared__ __attribute__((aligned(16))) float Bs[TB][ROW];
  __shared__ __attribute__((aligned(16))) float Cs[TB][ROW];
  __shared__ __attribute__((aligned(16))) float dx[TB][PB];
  __shared__ __attribute__((aligned(16))) float ys[TB][PB + 1];  // padded: neighbouring lanes write neighbouring rows
  __shared__ float dts[LB], dAs[LB];
  const int s = blockIdx.x, h = blockIdx.y;
  const int sl = slot[s];
  const int t0 = cu[s], t1 = cu[s + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chunk = lane % CH, pl = wave * PW + lane / CH;
  const int p0 = blockIdx.z * PB;
  const int inner = nh * P, C = inner + 2 * G * N;
  if (sl < 0) {  // padding rows: defined output, no state
    for (int i = threadIdx.x; i < (t1 - t0) * PB; i += 256)
      if (p0 + i % PB < P) y[(long)(t0 + i / PB) * inner + (long)h * P + p0 + i % PB] = 0.f;
    return;
  }
  if (t1 <= t0) return;
  const int n0 = chunk * 8;
  const int g = h / (nh / G);
  float S[8];
  float* sp = state + (((long)sl * nh + h) * N) * P + p0 + pl;
  const bool carried = ctx[s] > 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) S[i] = (carried && p0 + pl < P && n0 + i < N) ? sp[(long)(n0 + i) * P] : 0.f;
  const bool fixed = decay != nullptr;  // fixed decay per head: dt = 1, no skip term
  const float A = fixed ? 0.f : expf(a_log[h]), Dh = fixed ? 0.f : d_skip[h], bias = fixed ? 0.f : dt_bias[h];
  const float dfix = fixed ? decay[h] : 0.f;
  const int boff = n0 + (n0 >> 6) * 4;
  Raw8<T> rb[NB], rc[NB];
  T rx[NX];
  auto fetch = [&](int tb) {  // tokens past the segment read its last row, states past N the last ones
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = threadIdx.x + 256 * u, n = i % CH * 8;
      const T* row = xbc + (long)min(tb + min(i / CH, TB - 1), t1 - 1) * C + inner + g * N;
      if (vec) {
        rb[u].from(row + min(n, N - 8));
        rc[u].from(row + G * N + min(n, N - 8));
      } else {
        rb[u].from(row, n, N - 1);
        rc[u].from(row + G * N, n, N - 1);
      }
    }
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int i = threadIdx.x + 256 * u;
      rx[u] = xbc[(long)min(tb + min(i / PB, TB - 1), t1 - 1) * C + (long)h * P + min(p0 + i % PB, P - 1)];
    }
  };
  struct Token {
    float b[8], c[8], d, dA;
  };
  auto stage = [&](Token& k, int tt, int lb) {  // one staged token into registers
    load8(&Bs[tt][boff], k.b);
    load8(&Cs[tt][boff], k.c);
    k.dA = dAs[lb + tt];
    k.d = dx[tt][pl];
  };
  auto token = [&](const Token& k) -> float {
#pragma unroll
    for (int i = 0; i < 8; ++i) S[i] = fmaf(S[i], k.dA, k.d * k.b[i]);
    float a = fmaf(S[0], k.c[0], S[1] * k.c[1]);
#pragma unroll
    for (int i = 2; i < 8; ++i) a = fmaf(S[i], k.c[i], a);
    return group_sum<CH>(a);
  };
  fetch(t0);
  for (int tb = t0; tb < t1; tb += TB) {
    const int nt = min(TB, t1 - tb), lb = (tb - t0) % LB;
    if (lb == 0) {  // the step sizes and decays of the next 256 tokens (all have left the loop over the last ones)
      const int t = min(tb + (int)threadIdx.x, t1 - 1);
      float dt = 1.f, dA = dfix;
      if (!fixed) {
        const float raw = ldf(proj + (long)t * p_stride + dt_col + h) + bias;
        dt = raw > 20.f ? raw : log1pf(expf(raw));
        dA = expf(-A * dt);
      }
      dts[threadIdx.x] = dt;
      dAs[threadIdx.x] = dA;
      __syncthreads();
    }
    float ex[NX];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = threadIdx.x + 256 * u, tt = i / CH, n = i % CH * 8;
      if (NB * 256 == TB * CH || i < TB * CH) {
        float fb[8], fc[8];
        rb[u].to(fb);
        rc[u].to(fc);
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // states beyond N stay zero
          fb[k] = n + k < N ? fb[k] : 0.f;
          fc[k] = n + k < N ? fc[k] : 0.f;
        }
        store8(&Bs[tt][n + (n >> 6) * 4], fb);
        store8(&Cs[tt][n + (n >> 6) * 4], fc);
      }
    }
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int i = threadIdx.x + 256 * u, tt = min(i / PB, TB - 1);
      ex[u] = ldf(&rx[u]);
      if (NX * 256 == TB * PB || i < TB * PB) dx[tt][i % PB] = dts[lb + tt] * ex[u];
    }
    __syncthreads();
    if (tb + TB < t1) fetch(tb + TB);
    if (nt == TB) {
      Token k[2];  // the next one is read while one is processed
      stage(k[0], 0, lb);
#pragma unroll
      for (int t4 = 0; t4 < TB; t4 += GR) {
        float keep = 0.f;
#pragma unroll
        for (int j = 0; j < GR; ++j) {
          if (t4 + j + 1 < TB) stage(k[(t4 + j + 1) & 1], t4 + j + 1, lb);
          __builtin_amdgcn_sched_barrier(0);  // (the reads would be moved down to their uses)
          const float acc = token(k[(t4 + j) & 1]);
          keep = chunk == j ? acc : keep;
        }
        if (CH <= TB || chunk < TB) ys[t4 + chunk][pl] = keep;
      }
    } else {
      for (int tt = 0; tt < nt; ++tt) {
        Token k;
        stage(k, tt, lb);
        const float acc = token(k);
        if (chunk == 0) ys[tt][pl] = acc;
      }
    }
    __syncthreads();  // the tile's inputs are consumed and its read-outs complete
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int i = threadIdx.x + 256 * u, tt = i / PB, p = p0 + i % PB;
      if (tt < nt && p < P) y[(long)(tb + tt) * inner + (long)h * P + p] = fmaf(Dh, ex[u], ys[tt][i % PB]);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (p0 + pl < P && n0 + i < N) sp[(long)(n0 + i) * P] = S[i];
}

// The same with the products dt x (x) B taken off the vector unit, which the mapping above keeps busy all the time, and the sums the
// same bit for bit: a wave holds 64 states of 16 values of p, and v_mfma_f32_16x16x1 (four blocks, no sum: each of its results is
// one rounded product) writes the products of a token.  Row r of block k is the wave's state 16 (r / 4) + 4 k + r % 4, so that
// quarter q of the wave holds states 16 q .. 16 q + 15, each eight of which in neighbouring registers, and the sums over eight meet
// in the order of the mapping above: inside a lane, between the quarters, then between the NW = N / 64 waves that share a p, whose
// read-outs meet in LDS.  Per token a lane is left with two instructions per state; the products of a token are formed while the
// one before runs, its B and dt x read one token earlier still.  Rows past the segment's end are staged as zeros with decay 1,
// which leave the state as it is.  A wave alone on a SIMD issues every eighth cycle here, two of them every fifth, hence no more
// than 64 states to a wave: with 128 of them four prompts of 2048 tokens (64 heads of 64 x 128) took 585 us, so 464; one prompt
// 294 (758 before either mapping was reworked).
template <typename T, int NW>
__global__ __launch_bounds__(256, 2) void ssm_scan_tile_kernel(float* __restrict__ y, const T* __restrict__ xbc,
                                                               const T* __restrict__ proj, long p_stride, int dt_col,
                                                               const float* __restrict__ dt_bias,
                                                               const float* __restrict__ a_log,
                                                               const float* __restrict__ d_skip,
                                                               const float* __restrict__ decay,
                                                               float* __restrict__ state, const int* __restrict__ cu,
                                                               const int* __restrict__ ctx, const int* __restrict__ slot,
                                                               int nh, int P, int N, int G) {
  typedef float floatx16 __attribute__((ext_vector_type(16)));
  constexpr int TB = NW < 4 ? 32 : 16, PB = 64 / NW, LB = 256, NS = 64 * NW, CR = NS / 8, XR = PB / 4;
  constexpr int ROW = NS / 16 * 20;  // state n sits at n + 4 (n / 16): the quarters' reads 20 banks apart
  constexpr int NB = TB * CR / 256, NX = (TB * XR + 255) / 256;
  __shared__ __attribute__((aligned(16))) float Bs[TB][ROW];
  __shared__ __attribute__((aligned(16))) float Cs[TB][ROW];
  __shared__ __attribute__((aligned(16))) float dx[TB][PB];
  __shared__ __attribute__((aligned(16))) float ys[NW][TB][PB + 16];
  __shared__ float dts[LB], dAs[LB];
  const int s = blockIdx.x, h = blockIdx.y;
  const int sl = slot[s];
  const int t0 = cu[s], t1 = cu[s + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, wn = wave % NW;
  const int pl = wave / NW * 16 + (lane & 15), p0 = blockIdx.z * PB, p = p0 + pl;
  const int inner = nh * P, C = inner + 2 * G * N;
  const int xp = threadIdx.x % XR * 4, xt0 = threadIdx.x / XR;  // staging, finishing: values xp .. xp + 3 of tokens xt0 + 256 / XR u
  if (sl < 0) {  // padding rows: defined output, no state
    if (p0 + xp < P)
      for (int t = t0 + xt0; t < t1; t += 256 / XR)
        *reinterpret_cast<float4*>(y + (long)t * inner + (long)h * P + p0 + xp) = make_float4(0.f, 0.f, 0.f, 0.f);
    return;
  }
  if (t1 <= t0) return;
  const int g = h / (nh / G);
  float S[16];
  float* sp = state + (((long)sl * nh + h) * N) * P + p;
  const bool carried = ctx[s] > 0 && p < P;
  const int n0 = 64 * wn + 16 * q;
#pragma unroll
  for (int i = 0; i < 16; ++i) S[i] = carried && n0 + i < N ? sp[(long)(n0 + i) * P] : 0.f;
  const bool fixed = decay != nullptr;  // fixed decay per head: dt = 1, no skip term
  const float A = fixed ? 0.f : expf(a_log[h]), Dh = fixed ? 0.f : d_skip[h], bias = fixed ? 0.f : dt_bias[h];
  const float dfix = fixed ? decay[h] : 0.f;
  const int coff = 80 * wn + 20 * q;                                          // this quarter's states
  const int aoff = 80 * wn + 20 * ((lane & 15) >> 2) + 4 * q + (lane & 3);    // this lane's row of the product
  Raw8<T> rb[NB], rc[NB];
  T rx[NX][4];
  auto fetch = [&](int tb) {
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = threadIdx.x + 256 * u, n = min(i % CR * 8, N - 8);
      const T* row = xbc + (long)min(tb + i / CR, t1 - 1) * C + inner + g * N + n;
      rb[u].from(row);
      rc[u].from(row + G * N);
    }
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const T* row = xbc + (long)min(tb + xt0 + 256 / XR * u, t1 - 1) * C + (long)h * P + min(p0 + xp, P - 4);
      __builtin_memcpy(rx[u], __builtin_assume_aligned(row, 4 * sizeof(T)), 4 * sizeof(T));
    }
  };
  struct Ab {
    float a, d, dA;
  };
  auto read_ab = [&](Ab& k, int tt, int lb) {
    k.a = Bs[tt][aoff];
    k.d = dx[tt][pl];
    k.dA = dAs[lb + tt];
  };
  auto read_c = [&](float (&c)[16], int tt) {
    load8(&Cs[tt][coff], &c[0]);
    load8(&Cs[tt][coff + 8], &c[8]);
  };
  auto products = [&](const Ab& k) {
    const floatx16 zero = {};
    return __builtin_amdgcn_mfma_f32_16x16x1f32(k.a, k.d, zero, 0, 0, 0);
  };
  fetch(t0);
  for (int tb = t0; tb < t1; tb += TB) {
    const int nt = min(TB, t1 - tb), lb = (tb - t0) % LB;
    if (lb == 0) {  // the step sizes and decays of the next 256 tokens (all have left the loop over the last ones)
      const int t = tb + (int)threadIdx.x;
      float dt = 1.f, dA = dfix;
      if (!fixed) {
        const float raw = ldf(proj + (long)min(t, t1 - 1) * p_stride + dt_col + h) + bias;
        dt = raw > 20.f ? raw : log1pf(expf(raw));
        dA = expf(-A * dt);
      }
      dts[threadIdx.x] = dt;
      dAs[threadIdx.x] = t < t1 ? dA : 1.f;
      __syncthreads();
    }
    float ex[NX][4];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = threadIdx.x + 256 * u, tt = i / CR, n = i % CR * 8;
      float fb[8], fc[8];
      rb[u].to(fb);
      rc[u].to(fc);
      const bool in = n < N && tt < nt;  // (N is a multiple of 8)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        fb[k] = in ? fb[k] : 0.f;
        fc[k] = in ? fc[k] : 0.f;
      }
      store8(&Bs[tt][n + 4 * (n / 16)], fb);
      store8(&Cs[tt][n + 4 * (n / 16)], fc);
    }
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int xt = xt0 + 256 / XR * u;
#pragma unroll
      for (int v = 0; v < 4; ++v) ex[u][v] = ldf(&rx[u][v]);
      if (256 / XR * NX == TB || xt < TB) {
        const float dt = dts[lb + xt];
        *reinterpret_cast<float4*>(&dx[xt][xp]) = xt < nt ? make_float4(dt * ex[u][0], dt * ex[u][1], dt * ex[u][2], dt * ex[u][3])
                                                          : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
    __syncthreads();
    if (tb + TB < t1) fetch(tb + TB);
    Ab ab[2];
    float c[2][16];
    floatx16 t[2];
    read_ab(ab[0], 0, lb);
    read_ab(ab[1], 1, lb);
    read_c(c[0], 0);
    t[0] = products(ab[0]);
    float dA[2] = {ab[0].dA, 0.f}, r[4];
#pragma unroll
    for (int tt = 0; tt < TB; ++tt) {
      if (tt + 1 < TB) {
        read_c(c[(tt + 1) & 1], tt + 1);
        t[(tt + 1) & 1] = products(ab[(tt + 1) & 1]);
        dA[(tt + 1) & 1] = ab[(tt + 1) & 1].dA;
      }
      if (tt + 2 < TB) read_ab(ab[tt & 1], tt + 2, lb);
      __builtin_amdgcn_sched_barrier(0);  // (the reads would be moved down to their uses)
#pragma unroll
      for (int i = 0; i < 16; ++i) S[i] = fmaf(S[i], dA[tt & 1], t[tt & 1][i]);
      float a[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const float* cv = &c[tt & 1][8 * m];
        a[m] = fmaf(S[8 * m], cv[0], S[8 * m + 1] * cv[1]);
#pragma unroll
        for (int i = 2; i < 8; ++i) a[m] = fmaf(S[8 * m + i], cv[i], a[m]);
      }
      r[tt & 3] = a[0] + a[1];
      if ((tt & 3) == 3) {  // four tokens' sums over the quarters in three exchanges: quarter k ends with token k's
        const float r01 = swap16_sum(r[0], r[1]), r23 = swap16_sum(r[2], r[3]);
        ys[wn][tt - 3 + q][pl] = swap32_sum(r01, r23);
      }
    }
    __syncthreads();  // the tile's inputs are consumed and its read-outs complete
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int xt = xt0 + 256 / XR * u;
      if (xt >= nt || p0 + xp >= P) continue;
      float o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        o[v] = ys[0][xt][xp + v];
        if (NW == 2) o[v] += ys[NW - 1][xt][xp + v];
        if (NW == 4) o[v] = (o[v] + ys[1 % NW][xt][xp + v]) + (ys[2 % NW][xt][xp + v] + ys[3 % NW][xt][xp + v]);
        o[v] = fmaf(Dh, ex[u][v], o[v]);
      }
      *reinterpret_cast<float4*>(y + (long)(tb + xt) * inner + (long)h * P + p0 + xp) = make_float4(o[0], o[1], o[2], o[3]);
    }
  }
  if (p < P)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (n0 + i < N) sp[(long)(n0 + i) * P] = S[i];
}

}  // namespace k8sllm

using namespace k8sllm;

// one token a segment, rows that the step kernel can read four values at a time (some: groups behind the last repeat it)
template <typename T>
static bool step_sizes(const void* xbc, const float* state, int P, int N) {
  return P % 4 == 0 && N % 4 == 0 && N > 0 && N <= 256 && reinterpret_cast<uintptr_t>(state) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(xbc) % (4 * sizeof(T)) == 0;
}
template <typename T>
static int launch_step(float* y, const void* xbc, long x_stride, int silu, const void* proj, long p_stride, int dt_col, const float* dt_bias,
                       const float* a_log, const float* d_skip, const float* decay, float* state, const int* cu, const int* ctx,
                       const int* slot, int S, int nh, int P, int N, int G, hipStream_t s) {
  const dim3 grid((unsigned)S, (unsigned)nh, (unsigned)((P + 63) / 64));
  const bool once = 4l * S * nh * N * P > kStateOnceBytes;
#define K8SLLM_STEP(NPT)                                                                                                 \
  hipLaunchKernelGGL((once ? &ssm_step_kernel<T, NPT, true> : &ssm_step_kernel<T, NPT, false>), grid, dim3(256), 0, s, y,  \
                     (const T*)xbc, (const T*)proj, p_stride, dt_col, dt_bias, a_log, d_skip, decay, state, cu, ctx, slot, nh, \
                     P, N, G, x_stride, silu)
  if (N <= 16) K8SLLM_STEP(4);
  else if (N <= 32) K8SLLM_STEP(8);
  else if (N <= 64) K8SLLM_STEP(16);
  else if (N <= 128) K8SLLM_STEP(32);
  else K8SLLM_STEP(64);
#undef K8SLLM_STEP
  return (int)hipGetLastError();
}

template <typename T>
static int launch_scan(float* y, const void* xbc, const void* proj, long p_stride, int dt_col, const float* dt_bias,
                       const float* a_log, const float* d_skip, const float* decay, float* state, const int* cu, const int* ctx,
                       const int* slot, int S, int nh, int P, int N, int G, int wide, int step, hipStream_t s) {
  if (wide && N > 8) {  // long segments: 8 states per lane
    const int vec = N % 8 == 0 && (nh * P) % 8 == 0 && reinterpret_cast<uintptr_t>(xbc) % 16 == 0;
    // the tile form wants 16-byte rows of B and C and 4 values of p at a time; below 33 states half its products would be padding
    if (N > 32 && vec && P % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0) {
#define K8SLLM_TILE(NW)                                                                                              \
  hipLaunchKernelGGL((ssm_scan_tile_kernel<T, NW>),                                                                   \
                     dim3((unsigned)S, (unsigned)nh, (unsigned)((P + 64 / NW - 1) / (64 / NW))), dim3(256), 0, s, y,   \
                     (const T*)xbc, (const T*)proj, p_stride, dt_col, dt_bias, a_log, d_skip, decay, state, cu, ctx, slot, nh, \
                     P, N, G)
      if (N <= 64) K8SLLM_TILE(1);
      else if (N <= 128) K8SLLM_TILE(2);
      else if (N <= 256) K8SLLM_TILE(4);
      else return -1;
#undef K8SLLM_TILE
      return (int)hipGetLastError();
    }
#define K8SLLM_WIDE(CH)                                                                                              \
  hipLaunchKernelGGL((ssm_scan_wide_kernel<T, CH>), dim3((unsigned)S, (unsigned)nh, (unsigned)((P + 256 / CH - 1) / (256 / CH))), \
                     dim3(256), 0, s, y, (const T*)xbc, (const T*)proj, p_stride, dt_col, dt_bias, a_log, d_skip, decay, state, \
                     cu, ctx, slot, nh, P, N, G, vec)
    if (N <= 16) K8SLLM_WIDE(2);
    else if (N <= 32) K8SLLM_WIDE(4);
    else if (N <= 64) K8SLLM_WIDE(8);
    else if (N <= 128) K8SLLM_WIDE(16);
    else if (N <= 256) K8SLLM_WIDE(32);
    else return -1;
#undef K8SLLM_WIDE
    return (int)hipGetLastError();
  }
  const dim3 grid((unsigned)S, (unsigned)nh, (unsigned)((P + 63) / 64));
  if (step && step_sizes<T>(xbc, state, P, N))
    return launch_step<T>(y, xbc, nh * P + 2l * G * N, 0, proj, p_stride, dt_col, dt_bias, a_log, d_skip, decay, state, cu, ctx, slot, S, nh,
                          P, N, G, s);
#define K8SLLM_SCAN(NPT)                                                                                              \
  hipLaunchKernelGGL((ssm_scan_kernel<T, NPT>), grid, dim3(256), 0, s, y, (const T*)xbc, (const T*)proj, p_stride,    \
                     dt_col, dt_bias, a_log, d_skip, decay, state, cu, ctx, slot, nh, P, N, G)
  if (N <= 16) K8SLLM_SCAN(4);
  else if (N <= 32) K8SLLM_SCAN(8);
  else if (N <= 64) K8SLLM_SCAN(16);
  else if (N <= 128) K8SLLM_SCAN(32);
  else if (N <= 256) K8SLLM_SCAN(64);
  else return -1;
#undef K8SLLM_SCAN
  return (int)hipGetLastError();
}

template <typename T>
static int launch_conv(void* out, const void* proj, long stride, int col0, int C, const float* cw, const float* cb, int taps,
                       void* state, const int* cu, const int* ctx, const int* slot, int S, long rows, hipStream_t s) {
  const int gy = (C + 255) / 256, gy8 = (C / 8 + 255) / 256;
  if (rows <= S && taps == 4 && C % 8 == 0 && col0 % 8 == 0 && stride % 8 == 0) {
    hipLaunchKernelGGL(conv_step_kernel<T>, dim3((unsigned)S, (unsigned)gy8), dim3(256), 0, s, (T*)out, (const T*)proj, stride, col0, C, cw, cb,
                       (T*)state, cu, ctx, slot);
    return (int)hipGetLastError();
  }
  if (C % 8 == 0 && col0 % 8 == 0 && stride % 8 == 0) {
#define K8SLLM_CONV(R)                                                                                                 \
  hipLaunchKernelGGL((conv_silu_vec8_kernel<T, R>), dim3((unsigned)((rows + R - 1) / R), (unsigned)gy8), dim3(256), 0, s, (T*)out, \
                     (const T*)proj, stride, col0, C, cw, cb, taps, (const T*)state, cu, ctx, slot, S, (int)rows)
    // four rows a thread from 512 rows on (773 of 4096 channels: 15.9 us one row a thread, 12.9 four), below them it lacks threads
    // (256: 9.6 / 10.6); eight or sixteen rows are no faster at 8000 and slower where segments start (13 prompts of 300: 43 us with
    // one row, 25 with four, 28 with eight)
    if (taps == 4 && rows >= 512) K8SLLM_CONV(4);
    else K8SLLM_CONV(1);
#undef K8SLLM_CONV
  } else {
    hipLaunchKernelGGL(conv_silu_kernel<T>, dim3((unsigned)rows, (unsigned)gy), dim3(256), 0, s, (T*)out, (const T*)proj, stride, col0,
                       C, cw, cb, taps, (const T*)state, cu, ctx, slot, S);
  }
  if (taps > 1)
    hipLaunchKernelGGL(conv_state_step_kernel<T>, dim3((unsigned)S, (unsigned)gy), dim3(256), 0, s, (T*)state, (const T*)proj, stride,
                       col0, C, taps, cu, ctx, slot);
  return (int)hipGetLastError();
}

extern "C" {

int k8sllm_hy_conv_silu(void* out, const void* proj, long stride, int col0, int C, const float* cw, const float* cb,
                        int taps, void* state, const int* cu, const int* ctx, const int* slot, int S, long T, int f32,
                        hipStream_t s) {
  if (T <= 0 || S <= 0) return 0;
  if (taps < 1 || taps > kMaxTaps) return -1;
  return f32 ? launch_conv<float>(out, proj, stride, col0, C, cw, cb, taps, state, cu, ctx, slot, S, T, s)
             : launch_conv<bf16_t>(out, proj, stride, col0, C, cw, cb, taps, state, cu, ctx, slot, S, T, s);
}

int k8sllm_hy_ssm_scan(float* y, const void* xbc, const void* proj, long p_stride, int dt_col, const float* dt_bias,
                       const float* a_log, const float* d_skip, const float* decay, float* state, const int* cu, const int* ctx,
                       const int* slot, int S, long T, int nh, int P, int N, int G, int f32, int mode, hipStream_t s) {
  if (S <= 0) return 0;
  if (G < 1 || nh % G) return -1;
  // mode 0: by the step's mean segment length (prompts: the thin mapping; one token each: the step kernel); 1 / 2: forced (tests)
  const int wide = mode == 2 || (mode == 0 && T >= 32L * S), step = mode == 0 && T <= S;
  if (decay == nullptr && (proj == nullptr || dt_bias == nullptr || a_log == nullptr || d_skip == nullptr)) return -1;
  return f32 ? launch_scan<float>(y, xbc, proj, p_stride, dt_col, dt_bias, a_log, d_skip, decay, state, cu, ctx, slot,
                                  S, nh, P, N, G, wide, step, s)
             : launch_scan<bf16_t>(y, xbc, proj, p_stride, dt_col, dt_bias, a_log, d_skip, decay, state, cu, ctx, slot,
                                   S, nh, P, N, G, wide, step, s);
}

// Linear attention of one token a segment (T <= S), v, k and q the SiLU of a projection's first columns, rows x_stride apart.  1: not these sizes.
int k8sllm_hy_linear_step(float* y, const void* proj, long x_stride, const float* decay, float* state, const int* cu, const int* ctx,
                          const int* slot, int S, int H, int dk, int dv, int f32, hipStream_t s) {
  if (S <= 0) return 0;
  if (x_stride % 4 || !(f32 ? step_sizes<float>(proj, state, dv, dk) : step_sizes<bf16_t>(proj, state, dv, dk))) return 1;
  return f32 ? launch_step<float>(y, proj, x_stride, 1, nullptr, 0, 0, nullptr, nullptr, nullptr, decay, state, cu, ctx, slot, S, H, dv, dk, H, s)
             : launch_step<bf16_t>(y, proj, x_stride, 1, nullptr, 0, 0, nullptr, nullptr, nullptr, decay, state, cu, ctx, slot, S, H, dv, dk, H, s);
}
}
