// The selective state-space recurrence with a decay per channel AND state (any channel count, up to 256
// states; everything from the step sizes on fp32).  Per segment, channel c and state n, token by token:
//     dt = softplus(dt_raw[t][c] + dt_bias[c])
//     S[c][n] <- exp(-exp(a_log[c][n]) dt) S[c][n] + dt x_t[c] B_t[n]
//     y_t[c]  = sum_n S[c][n] C_t[n] + D[c] x_t[c];      out_t[c] = y_t[c] * silu(z_t[c])
// The state slot [C][N] is read at the segment's start (zero for a sequence that starts in this step) and
// written back at its end.  A segment is one sequence's rows of this step: cu[s] .. cu[s+1], ctx[s] tokens
// already in its state, slot[s] its state slot (< 0: padding rows, output zero).
//
// Workgroup = 4 waves = (segment, 256 / LPC channels).  A channel is owned by LPC neighbouring lanes, each
// with NPL of its states (and their exponents' factors) in registers; the read-out's partial sums are DPP adds
// over those lanes.  16 tokens at a time are staged in LDS: step sizes after softplus, dt x, B, C; the raw
// values of the next 16 are fetched into registers while the current ones are processed.  The read-outs of
// a tile meet in LDS (a lane keeps every LPC-th one, so LPC tokens need one LDS write), and the whole
// workgroup adds the skip term, applies the gate and stores rows.  Loads are not predicated: a token past
// the segment reads the segment's last row, a channel past the end the last channel, and what they must
// not contribute is zeroed when it is staged - a branch around a load would wait for it there.
// One exponential per state and token (v_exp_f32 in base 2, log2 e folded into the factor) bounds a wave, and the chain of
// tokens a launch with few sequences: there long segments are cut into spans of 128 or 256 tokens that run side by side (MODE
// kSpanEnds, then kSpanRun).  The first launch runs every span but a segment's last from a zero state and keeps its end E and
// its sum of step sizes s; since a span's decays multiply to exp(-exp(a_log) s), the state before span k is
//     I;  then for j = 0 .. k - 1:  S <- exp(-exp(a_log) s_j) S + E_j
// which the second launch folds in front of its own tokens (I, the state the segment starts from, is kept in the last span's
// place, so that no workgroup reads the slot that another one writes).  One prompt of 8192 tokens, 4096 channels x 16 states:
// 1072 us whole, 290 in spans, each launch at the rate of its exponentials and multiply-adds; 2048 tokens 265 -> 86.
#include "chunk_seg.h"

namespace k8sllm {

// log(1 + exp(x)) to a few units in the last place without the library's branches: max(x, 0) + log1p(e),
// e = exp(-|x|); log1p by its series below 1/32, by v_log_f32 above
__device__ __forceinline__ float softplus_fast(float x) {
  const float a = -fabsf(x), t = a * 1.44269504088896341f;
  const float lo = fmaf(a, 1.44269504088896341f, -t);  // what rounding the product dropped
  const float e2 = __builtin_amdgcn_exp2f(t), e = fmaf(e2, lo * 0.693147180559945309f, e2);
  const float series = e * fmaf(e, fmaf(e, fmaf(e, -0.25f, 0.333333333f), -0.5f), 1.f);
  const float lg = __builtin_amdgcn_logf(1.f + e) * 0.693147180559945309f;
  return fmaxf(x, 0.f) + (e < 0.03125f ? series : lg);
}

template <typename T, int LPC, int NPL, int MODE>
__global__ __launch_bounds__(256) void selective_scan_kernel(
    T* __restrict__ out, const T* __restrict__ xc, const T* __restrict__ q, long q_stride, int b_col, int c_col,
    const T* __restrict__ dt, long dt_stride, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
    const float* __restrict__ d_skip, const T* __restrict__ z, long z_stride, float* __restrict__ state,
    const int* __restrict__ cu, const int* __restrict__ ctx, const int* __restrict__ slot, int n_seg, int span, int C, int N,
    float* __restrict__ ends, float* __restrict__ sums) {
  constexpr int TB = 16, PB = 256 / LPC, NS = LPC * NPL;
  constexpr int NV = TB * PB / 256;           // (token, channel) pairs a thread stages and finishes
  constexpr int NB = (TB * NS + 255) / 256;   // B / C elements a thread stages
  __shared__ __attribute__((aligned(16))) float Bs[TB][NS];
  __shared__ __attribute__((aligned(16))) float Cs[TB][NS];
  __shared__ float dts[TB][PB], us[TB][PB];
  __shared__ float ys[TB][PB + 64 / LPC];  // padded: the lanes of a channel write neighbouring rows to different banks
  ChunkAt at = {0, 0, 0, 0, 1};
  SegAt own;
  int by = blockIdx.y;  // which channels
  if (MODE == kWhole) {
    // (segments side by side within a round: an XCD has few of them, whose tokens its L2 then holds for all channels)
    const int i = blockIdx.x + gridDim.x * blockIdx.y, groups = gridDim.y, round = min(max(1, 256 / groups), n_seg);
    const int k = i / (round * groups), j = i - k * round * groups, m = min(round, n_seg - k * round);
    by = j / m;
    own = segment_in_turn(cu, slot, n_seg, k * round + j - by * m, groups, 1 << 30);
    at.seg = own.seg;
  } else {
    at = chunk_at(cu, n_seg, blockIdx.x, span);
    if (at.seg < 0) return;
    own = {at.seg, slot[at.seg], at.row, at.row + at.n};
    if (MODE == kSpanEnds && (at.k == at.count - 1 || own.slot < 0)) return;
  }
  const int s = own.seg, sl = own.slot, t0 = own.t0, t1 = own.t1;
  const int pc = threadIdx.x % PB, tt0 = threadIdx.x / PB;  // staging: channel pc, tokens tt0 + LPC u
  const int cs = by * PB + pc;
  const bool slive = cs < C;
  if (sl < 0) {  // padding rows: defined output, no state
    if (slive)
      for (int t = t0 + tt0; t < t1; t += LPC) stf(out + (long)t * C + cs, 0.f);
    return;
  }
  if (t1 <= t0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chunk = lane % LPC, pl = wave * (64 / LPC) + lane / LPC;
  const int c = by * PB + pl, n0 = chunk * NPL;
  const bool live = c < C;
  const bool vec = (N & 3) == 0 && n0 + NPL <= N;
  const bool carried = ctx[s] > 0 && (MODE == kWhole || at.count == 1 || (MODE == kSpanEnds && at.k == 0));
  float S[NPL], A[NPL];
  float* sp = state + ((long)sl * C + c) * N + n0;
  const float* ap = a_log + (long)c * N + n0;
  if (live && vec) {
#pragma unroll
    for (int i = 0; i < NPL; i += 4) {
      const float4 a = *reinterpret_cast<const float4*>(ap + i);
      A[i] = a.x; A[i + 1] = a.y; A[i + 2] = a.z; A[i + 3] = a.w;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (carried) v = *reinterpret_cast<const float4*>(sp + i);
      S[i] = v.x; S[i + 1] = v.y; S[i + 2] = v.z; S[i + 3] = v.w;
    }
#pragma unroll
    for (int i = 0; i < NPL; ++i) A[i] = -expf(A[i]) * 1.44269504088896341f;
  } else {
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      const bool in = live && n0 + i < N;
      A[i] = in ? -expf(ap[i]) * 1.44269504088896341f : 0.f;
      S[i] = (in && carried) ? sp[i] : 0.f;
    }
  }
  // span j's end state of this channel; the state that a segment of several spans starts from goes to the last one's place
  auto end_of = [&](int j) { return ends + (((long)blockIdx.x - at.k + j) * C + min(c, C - 1)) * N; };
  auto read = [&](float (&v)[NPL], const float* p) {
#pragma unroll
    for (int i = 0; i < NPL; i += 4) {
      if (vec) {
        const float4 f = *reinterpret_cast<const float4*>(p + n0 + i);
        v[i] = f.x; v[i + 1] = f.y; v[i + 2] = f.z; v[i + 3] = f.w;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[i + j] = p[min(n0 + i + j, N - 1)];
      }
    }
  };
  if (MODE == kSpanEnds && at.k == 0) {
    float* ip = end_of(at.count - 1);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      if (live && n0 + i < N) ip[n0 + i] = S[i];
      S[i] = 0.f;
    }
  }
  if (MODE == kSpanRun && at.count > 1) {
    read(S, end_of(at.count - 1));
#pragma unroll 4
    for (int j = 0; j < at.k; ++j) {
      float E[NPL];
      read(E, end_of(j));
      const float d = sums[((long)blockIdx.x - at.k + j) * C + min(c, C - 1)];
#pragma unroll
      for (int i = 0; i < NPL; ++i) S[i] = __builtin_amdgcn_exp2f(d * A[i]) * S[i] + E[i];
    }
#pragma unroll
    for (int i = 0; i < NPL; ++i)
      if (n0 + i >= N) S[i] = 0.f;
  }
  float dsum = 0.f;
  const float bias = slive ? dt_bias[cs] : 0.f, D = slive ? d_skip[cs] : 0.f;
  T rd[NV], rx[NV], rz[NV], rB[NB], rC[NB];
  const int cl = min(cs, C - 1);
  auto fetch = [&](int tb) {
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const long t = min(tb + tt0 + LPC * u, t1 - 1);
      rd[u] = dt[t * dt_stride + cl];
      rx[u] = xc[t * C + cl];
      if (MODE != kSpanEnds) rz[u] = z[t * z_stride + cl];
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = threadIdx.x + 256 * u;
      const T* row = q + (long)min(tb + i / NS, t1 - 1) * q_stride + min(i % NS, N - 1);
      rB[u] = row[b_col];
      if (MODE != kSpanEnds) rC[u] = row[c_col];
    }
  };
  auto token = [&](int tt) -> float {  // the recurrence for one staged token; the channel's read-out on all its lanes
    const float d = dts[tt][pl], u = us[tt][pl];
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < NPL; i += 4) {
      const float4 b = *reinterpret_cast<const float4*>(&Bs[tt][n0 + i]);
      float4 g;
      if (MODE != kSpanEnds) g = *reinterpret_cast<const float4*>(&Cs[tt][n0 + i]);
      S[i] = __builtin_amdgcn_exp2f(d * A[i]) * S[i] + u * b.x;
      S[i + 1] = __builtin_amdgcn_exp2f(d * A[i + 1]) * S[i + 1] + u * b.y;
      S[i + 2] = __builtin_amdgcn_exp2f(d * A[i + 2]) * S[i + 2] + u * b.z;
      S[i + 3] = __builtin_amdgcn_exp2f(d * A[i + 3]) * S[i + 3] + u * b.w;
      if (MODE != kSpanEnds) acc += S[i] * g.x + S[i + 1] * g.y + S[i + 2] * g.z + S[i + 3] * g.w;
    }
    if (MODE == kSpanEnds) {
      dsum += d;
      return 0.f;
    }
    return lanes_sum<LPC>(acc);
  };
  fetch(t0);
  for (int tb = t0; tb < t1; tb += TB) {
    const int nt = min(TB, t1 - tb);
    float ex[NV], ez[NV];  // this tile's x and gate, for its epilogue
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int tt = tt0 + LPC * u;
      const float d = softplus_fast(ldf(&rd[u]) + bias);
      ex[u] = ldf(&rx[u]);
      if (MODE != kSpanEnds) ez[u] = ldf(&rz[u]);
      dts[tt][pc] = d;
      us[tt][pc] = d * ex[u];
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = threadIdx.x + 256 * u;
      const bool in = i % NS < N;  // states beyond N stay zero
      if (NB * 256 == TB * NS || i < TB * NS) {
        (&Bs[0][0])[i] = in ? ldf(&rB[u]) : 0.f;
        if (MODE != kSpanEnds) (&Cs[0][0])[i] = in ? ldf(&rC[u]) : 0.f;
      }
    }
    __syncthreads();
    if (tb + TB < t1) fetch(tb + TB);
    if (MODE == kSpanEnds) {  // whole tiles: a span that is not its segment's last holds `span` tokens
#pragma unroll
      for (int tt = 0; tt < TB; ++tt) token(tt);
      __syncthreads();
      continue;
    }
    if (nt == TB) {
#pragma unroll
      for (int t4 = 0; t4 < TB; t4 += LPC) {
        float keep = 0.f;
#pragma unroll
        for (int j = 0; j < LPC; ++j) {
          const float acc = token(t4 + j);
          keep = chunk == j ? acc : keep;
        }
        ys[t4 + chunk][pl] = keep;
      }
    } else {
      for (int tt = 0; tt < nt; ++tt) {
        const float acc = token(tt);
        if (chunk == 0) ys[tt][pl] = acc;
      }
    }
    __syncthreads();  // the tile's inputs are consumed and its read-outs complete
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int tt = tt0 + LPC * u;
      if (slive && tt < nt) stf(out + (long)(tb + tt) * C + cs, (ys[tt][pc] + D * ex[u]) * silu_f(ez[u]));
    }
  }
  if (MODE == kSpanEnds) {
    sp = end_of(at.k) + n0;
    if (live && chunk == 0) sums[(long)blockIdx.x * C + c] = dsum;
  }
  if (live && (MODE != kSpanRun || at.k == at.count - 1)) {
    if (vec) {
#pragma unroll
      for (int i = 0; i < NPL; i += 4) *reinterpret_cast<float4*>(sp + i) = make_float4(S[i], S[i + 1], S[i + 2], S[i + 3]);
    } else {
#pragma unroll
      for (int i = 0; i < NPL; ++i)
        if (n0 + i < N) sp[i] = S[i];
    }
  }
}

// Steps of one token a segment (decode): a pass over the states, a channel on the lanes that selective_scan_kernel has for it, without
// its tiles of tokens in LDS.  The same operations in the same order: the same bits.  us, selective_scan_kernel / here: 8192 channels x 16, 1 segment 3.6 /
// 3.1, 16 8.9 / 6.1, 64 30.6 / 18.7, 128 54 / 31 (4.3 TB/s).
template <typename T, int LPC, int NPL, bool ONCE>
__global__ __launch_bounds__(256) void selective_step_kernel(
    T* __restrict__ out, const T* __restrict__ xc, const T* __restrict__ q, long q_stride, int b_col, int c_col,
    const T* __restrict__ dt, long dt_stride, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
    const float* __restrict__ d_skip, const T* __restrict__ z, long z_stride, float* __restrict__ state,
    const int* __restrict__ cu, const int* __restrict__ ctx, const int* __restrict__ slot, int C, int N) {
  constexpr int PB = 256 / LPC;
  const int s = blockIdx.x, sl = slot[s], t0 = cu[s], t1 = cu[s + 1];
  const int chunk = threadIdx.x % LPC, c = blockIdx.y * PB + threadIdx.x / LPC, cc = min(c, C - 1);
  if (sl < 0) {  // padding rows: defined output, no state
    if (c < C && chunk == 0)
      for (int t = t0; t < t1; ++t) stf(out + (long)t * C + c, 0.f);
    return;
  }
  if (t1 <= t0) return;
  const bool live = chunk * NPL < N;  // lanes behind the last state: the last ones again, counted as zero
  const int n0 = live ? chunk * NPL : N - NPL;
  float* sp = state + ((long)sl * C + cc) * N + n0;
  const float* ap = a_log + (long)cc * N + n0;
  const bool carried = ctx[s] > 0;
  float S[NPL], A[NPL];
#pragma unroll
  for (int i = 0; i < NPL; i += 4) {
    const f32v4 v = load_state<ONCE>(sp + i);
    S[i] = v[0]; S[i + 1] = v[1]; S[i + 2] = v[2]; S[i + 3] = v[3];
    load4(ap + i, A + i);
  }
  const float bias = dt_bias[cc], D = d_skip[cc];
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    A[i] = -expf(A[i]) * 1.44269504088896341f;
    S[i] = live && carried ? S[i] : 0.f;
  }
  for (int t = t0; t < t1; ++t) {
    const T* row = q + (long)t * q_stride + n0;
    float b[NPL], g[NPL];
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      b[i] = ldf(row + b_col + i);
      g[i] = ldf(row + c_col + i);
    }
    const float x = ldf(xc + (long)t * C + cc), zz = ldf(z + (long)t * z_stride + cc);
    const float d = softplus_fast(ldf(dt + (long)t * dt_stride + cc) + bias), u = d * x;
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < NPL; i += 4) {
#pragma unroll
      for (int j = i; j < i + 4; ++j) {
        S[j] = __builtin_amdgcn_exp2f(d * A[j]) * S[j] + u * b[j];
        S[j] = live ? S[j] : 0.f;
      }
      acc += S[i] * g[i] + S[i + 1] * g[i + 1] + S[i + 2] * g[i + 2] + S[i + 3] * g[i + 3];
    }
    acc = lanes_sum<LPC>(live ? acc : 0.f);
    if (c < C && chunk == 0) stf(out + (long)t * C + c, (acc + D * x) * silu_f(zz));
  }
  if (c < C && live) {
#pragma unroll
    for (int i = 0; i < NPL; i += 4) store_state<ONCE>(sp + i, f32v4{S[i], S[i + 1], S[i + 2], S[i + 3]});
  }
}

}  // namespace k8sllm

using namespace k8sllm;

static long channel_groups(int C, int N) {  // workgroups per segment or span
  const int lpc = N <= 8 ? 2 : N <= 16 ? 4 : N <= 64 ? 8 : 16;
  return (C + 256 / lpc - 1) / (256 / lpc);
}

// A span of 128 costs a workgroup 17 us and its longest fold grows with their number; from where spans of 256 give every
// compute unit four workgroups, these are faster (one prompt of 8192, 4096 channels x 16: 300 us against 321; of 2048: 111
// against 88).
static int span_tokens(long T, int C, int N) { return T * channel_groups(C, N) >= 256l * 1024 ? 256 : 128; }

template <typename T>
static int launch_selective(void* out, const void* xc, const void* q, long q_stride, int b_col, int c_col, const void* dt,
                            long dt_stride, const float* dt_bias, const float* a_log, const float* d_skip, const void* z,
                            long z_stride, float* state, const int* cu, const int* ctx, const int* slot, int S, int C,
                            int N, long T_, float* ws, int step, hipStream_t s) {
  const int span = span_tokens(T_, C, N);
  const long spans = T_ / span + S;
  float* sums = ws + spans * C * N;
#define K8SLLM_SSM(LPC, NPL, MODE)                                                                                           \
  hipLaunchKernelGGL((selective_scan_kernel<T, LPC, NPL, MODE>),                                                               \
                     dim3((unsigned)(MODE == kWhole ? S : spans), (unsigned)((C + 256 / LPC - 1) / (256 / LPC))), dim3(256), 0, s, \
                     (T*)out, (const T*)xc, (const T*)q, q_stride, b_col, c_col, (const T*)dt, dt_stride, dt_bias, a_log,       \
                     d_skip, (const T*)z, z_stride, state, cu, ctx, slot, S, span, C, N, ws, sums)
#define K8SLLM_ST(LPC, NPL)                                                                                                  \
  hipLaunchKernelGGL((4l * S * C * N > kStateOnceBytes ? &selective_step_kernel<T, LPC, NPL, true> : &selective_step_kernel<T, LPC, NPL, false>), \
                     dim3((unsigned)S, (unsigned)((C + 256 / LPC - 1) / (256 / LPC))), dim3(256), 0, s, (T*)out, (const T*)xc, \
                     (const T*)q, q_stride, b_col, c_col, (const T*)dt, dt_stride, dt_bias, a_log, d_skip, (const T*)z, z_stride, \
                     state, cu, ctx, slot, C, N)
  const bool whole = ((reinterpret_cast<uintptr_t>(state) | reinterpret_cast<uintptr_t>(a_log)) & 15) == 0;
#define K8SLLM_SS(LPC, NPL)                  \
  if (step && ws == nullptr && whole && N % NPL == 0) { \
    K8SLLM_ST(LPC, NPL);                     \
  } else if (ws != nullptr) {                \
    K8SLLM_SSM(LPC, NPL, kSpanEnds);         \
    K8SLLM_SSM(LPC, NPL, kSpanRun);          \
  } else {                                   \
    K8SLLM_SSM(LPC, NPL, kWhole);            \
  }
  if (N <= 8) { K8SLLM_SS(2, 4); }
  else if (N <= 16) { K8SLLM_SS(4, 4); }
  else if (N <= 32) { K8SLLM_SS(8, 4); }
  else if (N <= 64) { K8SLLM_SS(8, 8); }
  else if (N <= 128) { K8SLLM_SS(16, 8); }
  else if (N <= 256) { K8SLLM_SS(16, 16); }
  else return -1;
#undef K8SLLM_SS
#undef K8SLLM_ST
#undef K8SLLM_SSM
  return (int)hipGetLastError();
}

extern "C" {

// floats of workspace for a step of T rows in S segments, the longest of `longest` rows (0: not known, the mean is taken), that
// is to be cut into spans; 0: it runs whole (mode 1 / 2: whole / cut whatever the sizes).  Whole, a step takes as long as its
// longest segment's chain, 0.13 us a token, or as all its workgroups' tokens, 467 at a time; cut, twice the latter and what the
// spans' own chains and the folds come to, about 200 tokens' time.  Measured (4096 channels x 16, whole against cut): one
// prompt of 384 53 / 38 us, of 8192 1072 / 300; two of 4096 547 / 286; four of 2048 274 / 275; eight of 1024 211 / 287; one of
// 2048 beside 24 single tokens 322 / 115.
long k8sllm_hy_selective_scan_ws(long T, int S, int longest, int C, int N, int mode) {
  const long n = longest > 0 ? longest : S > 0 ? T / S : 0;
  const bool cut = mode == 2 || (mode == 0 && n >= 200 + T * channel_groups(C, N) / 233);
  return cut ? (T / span_tokens(T, C, N) + S) * C * (N + 1) : 0;
}

// xc, out [T][C] contiguous; q's rows hold B from b_col on and C from c_col on (N each); ws: nullptr, or the workspace of a
// step cut into spans; step: one token a segment may take the step kernel
int k8sllm_hy_selective_scan(void* out, const void* xc, const void* q, long q_stride, int b_col, int c_col,
                             const void* dt, long dt_stride, const float* dt_bias, const float* a_log, const float* d_skip,
                             const void* z, long z_stride, float* state, const int* cu, const int* ctx, const int* slot,
                             int S, long T, int C, int N, int f32, float* ws, int step, hipStream_t s) {
  if (S <= 0 || T <= 0) return 0;
  if (C < 1 || N < 1) return -1;
#define K8SLLM_ARGS \
  out, xc, q, q_stride, b_col, c_col, dt, dt_stride, dt_bias, a_log, d_skip, z, z_stride, state, cu, ctx, slot, S, C, N, T, ws, step && T <= S, s
  return f32 ? launch_selective<float>(K8SLLM_ARGS) : launch_selective<bf16_t>(K8SLLM_ARGS);
#undef K8SLLM_ARGS
}
}
