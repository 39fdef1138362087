// Linear attention with a decay per head and key channel, plain or with a bonus for the current token, bf16 prompts, in
// chunks of 64 tokens on the matrix cores (the recurrences are decay_scan.hip's).
//
// With L_i[c] the sum of log2 g[c] up to token i of the chunk and E_i = L_i (plain: a token reads the state behind its own
// decay and write) or L_(i-1) (bonus: the state before them):
//   O = Q' S_prev + M V        Q'_i[c] = q_i[c] 2^E_i[c],   M_ij = sum_c q_i[c] k_j[c] 2^(E_i[c] - L_j[c])  (j < i),
//                              M_ii = sum_c q_i[c] k_i[c] (plain; bonus: times w[c])
//   S = diag(2^L_n) S_prev + N V                                              N[c][j] = k_j[c] 2^(L_n[c] - L_j[c])
// No exponent is positive, so nothing overflows however fast a channel forgets: between sub-blocks of 16 tokens the
// exponent of M is split at the query block's first token, 2^(E_i - ref) 2^(ref - L_j), and inside a sub-block M is summed
// with running products of the decays, as the token-by-token form has them.
//  * decay_chunk_prep: a workgroup per (chunk, head), all in parallel, leaves Q', M and N as fp32 in operand order and 2^L_n in a
//    workspace.  Sums of log2 g are kept in 64 bits.
//  * decay_chunk_scan: eight waves per (segment, head, 16 NT value columns) walk the chunks, four for O, four for S; S is
//    published in LDS as three bf16 parts (split_bf16.h), double-buffered: one barrier per chunk.  The operands are split into
//    parts as they arrive.  Values are bf16 activations (exact), so their products take three instructions, Q' S the six that
//    matter at 2^-24.
//    Long segments that leave the chip idle are cut into spans of chunks: a launch for their ends, one for the outputs.
// What bounds it: the workspace's operands, 48 KiB per chunk and head at 64 channels, written once and read by every column
// block (as three bf16 parts they were 72 KiB, and the spans' second launch went at the rate of memory: 1 x 8000 rows, 32 heads of
// 64, both launches and the preparation 239 us, as fp32 221); the preparation also by vector instructions: it has no LDS read
// behind a branch, no branch per token, and reads the rows of a diagonal's next product ahead of this one's (268 -> 239 us).
// Measured, all launches (us, before these two changes; the staged scan with its preparation), 32 heads of 64 x 64 with a
// bonus: 1 x 8000 rows 221 (268; 1347), 4 x 2048 201 (250; 428); plain, 16 heads of 128 x 128: 1 x 8000 342 (457; 1548).  Error
// against 64 bits, 2048 rows, bonus: outputs 1.3e-7 (scan 2.7e-7), state 7.9e-8 (3.0e-7); plain: 2.3e-7 (1.5e-6), 2.1e-7 (2.0e-6).
#include "chunk_seg.h"
#include "split_bf16.h"
#include <type_traits>

namespace k8sllm {

// elements of Q', M and N of one (chunk, head) in the workspace
__host__ __device__ constexpr long kc_mats(int dk) { return 64L * (64 + 2 * dk); }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int KS, bool BONUS>
__global__ __launch_bounds__(256) void decay_chunk_prep_kernel(float* __restrict__ mats, float* __restrict__ ends,
                                                               const bf16_t* __restrict__ qkv, long stride, int q_col,
                                                               int k_col, const bf16_t* __restrict__ z, long z_stride,
                                                               const float* __restrict__ z_bias,
                                                               const float* __restrict__ a_log, float inv_tau, int dkind,
                                                               const float* __restrict__ bonus, const int* __restrict__ cu,
                                                               const int* __restrict__ slot, int S, int H, int Gk,
                                                               float q_scale) {
  constexpr int DK = 32 * KS, PK = DK + 8, PL = DK + 1, PG = DK + 4, PM = 68;  // (pitches under which sixteen rows lie in different banks)
  __shared__ __attribute__((aligned(16))) double Ll[64 * PL];  // L; later M as fp32 [64][PM]
  __shared__ __attribute__((aligned(16))) bf16_t Ql[64 * PK], Kl[64 * PK];
  __shared__ __attribute__((aligned(16))) float Gl[64 * PG];  // the decays
  float* Ml = reinterpret_cast<float*>(Ll);
  static_assert(64 * PM * 4 <= 64 * PL * 8 || KS == 1, "M fits where L was");
  __shared__ float Mx[KS == 1 ? 64 * PM : 1];
  __shared__ double Tl[256];
  const ChunkAt at = chunk_at(cu, S, blockIdx.x);
  if (at.seg < 0 || slot[at.seg] < 0) return;
  const int h = blockIdx.y, g = h / (H / Gk), n = at.n;
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, quad = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  {
    const int r = tid >> 2, c0 = (tid & 3) * (DK / 4);
    const bf16_t* row = qkv + (long)(at.row + min(r, n - 1)) * stride + (long)g * DK + c0;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      *reinterpret_cast<uint4*>(&Ql[r * PK + c0 + 8 * u]) = *reinterpret_cast<const uint4*>(row + q_col + 8 * u);
      *reinterpret_cast<uint4*>(&Kl[r * PK + c0 + 8 * u]) = *reinterpret_cast<const uint4*>(row + k_col + 8 * u);
    }
  }
  const float A = a_log != nullptr ? expf(a_log[h]) : 0.f;
  // decay sums: a thread takes a run of tokens of a channel (16, or 8 where 32 channels go at a time); the runs meet by
  // their totals
  constexpr int CT = DK % 64 == 0 ? 64 : 32, NQ = 256 / CT, QT = 64 / NQ;  // channels at a time, runs, tokens of a run
  const int cq = tid % CT, tq = tid / CT;
#pragma unroll
  for (int cb = 0; cb < DK; cb += CT) {
    const int c = cb + cq;
    bf16_t zr[QT];
#pragma unroll
    for (int i = 0; i < QT; ++i) zr[i] = z[(long)(at.row + min(QT * tq + i, n - 1)) * z_stride + (long)h * DK + c];
    const float zb = z_bias[(long)h * DK + c];
    float x[QT];
    double run = 0.0;
    auto decays = [&](auto kind) {  // (the kind's branch around the run, not around each token)
#pragma unroll
      for (int i = 0; i < QT; ++i) x[i] = log2_decay(bf2f(zr[i]) + zb, kind, A, inv_tau);
    };
    if (dkind == 0) decays(std::integral_constant<int, 0>{});
    else if (dkind == 1) decays(std::integral_constant<int, 1>{});
    else decays(std::integral_constant<int, 2>{});
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      const int t = QT * tq + i;
      x[i] = t < n ? x[i] : 0.f;
      Gl[t * PG + c] = __builtin_amdgcn_exp2f(x[i]);
      run += (double)x[i];
    }
    Tl[tq * CT + cq] = run;
    __syncthreads();
    double at_t = 0.0;
#pragma unroll
    for (int u = 0; u < NQ - 1; ++u) {
      const double v = Tl[u * CT + cq];
      at_t += u < tq ? v : 0.0;
    }
#pragma unroll
    for (int i = 0; i < QT; ++i) {
      at_t += (double)x[i];
      Ll[(QT * tq + i) * PL + c] = at_t;
    }
    __syncthreads();
  }
  const long ch = (long)blockIdx.x * H + h;
  float* Qo = mats + ch * kc_mats(DK);
  float* Mo = Qo + 64 * DK;
  float* No = Mo + 64 * 64;
  auto put = [&](float* o, int tile, const float* v) {  // a lane's eight values of a fragment, in two rows of 16 bytes a lane
#pragma unroll
    for (int k = 0; k < 2; ++k)
      *reinterpret_cast<float4*>(o + ((tile * 2 + k) * 64 + lane) * 4) = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
  };
  const int qi = 16 * w + c16, ei = qi - (BONUS ? 1 : 0);  // this lane's query; the token whose sum its reads carry
  // eight channels of a row: sums (zero before the first token) and activations
  auto sums8 = [&](int row, int c, double* d) {
    const double* l = Ll + max(row, 0) * PL + c;
#pragma unroll
    for (int i = 0; i < 8; ++i) d[i] = l[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) d[i] = row < 0 ? 0.0 : d[i];
  };
  auto acts8 = [&](const bf16_t* m, int row, int c, float* f) { unpack8(*reinterpret_cast<const uint4*>(&m[row * PK + c]), f); };
  // Q', and this query block's operand against earlier blocks, relative to the block's first token
  bf16x8 qf[KS][3];
  double ref[KS][8];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int c = 32 * ks + 8 * quad;
    double e[8], (&r)[8] = ref[ks];
    float q[8], a[8], b[8];
    sums8(ei, c, e);
    sums8(16 * w - 1, c, r);
    acts8(Ql, qi, c, q);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float qs = q[i] * q_scale;
      a[i] = qs * __builtin_amdgcn_exp2f((float)e[i]);
      b[i] = qs * __builtin_amdgcn_exp2f((float)(e[i] - r[i]));
    }
    put(Qo, w * KS + ks, a);
    uint32_t x[3][4];
    split_pairs<4>(b, x[0], x[1], x[2]);
#pragma unroll
    for (int k = 0; k < 3; ++k) qf[ks][k] = frag(x[k]);
  }
  // M against the earlier blocks: p[kt][i]: key 16 kt + 4 quad + i, query qi
  f32x4 p[3];
#pragma unroll
  for (int kt = 0; kt < 3; ++kt) {
    p[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (kt < w) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int c = 32 * ks + 8 * quad;
        const double (&r)[8] = ref[ks];
        double l[8];
        float k[8];
        sums8(16 * kt + c16, c, l);
        acts8(Kl, 16 * kt + c16, c, k);
#pragma unroll
        for (int i = 0; i < 8; ++i) k[i] *= __builtin_amdgcn_exp2f((float)(r[i] - l[i]));
        uint32_t x[3][4];
        split_pairs<4>(k, x[0], x[1], x[2]);
#pragma unroll
        for (int a = 2; a >= 0; --a)
#pragma unroll
          for (int b = 2 - a; b >= 0; --b) p[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(x[a]), qf[ks][b], p[kt], 0, 0, 0);
      }
    }
  }
  // N: rows are channels 16 rt + c16, eight tokens from 32 ks + 8 quad on
  for (int rt = w; rt < 2 * KS; rt += 4) {
    const int c = 16 * rt + c16;
    const double Ln = Ll[63 * PL + c];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int t = 32 * ks + 8 * quad + i;  // (the decay behind a token past the chunk is one)
        const uint32_t k = (uint32_t)Kl[t * PK + c] << 16;
        v[i] = __builtin_bit_cast(float, t < n ? k : 0u) * __builtin_amdgcn_exp2f((float)(Ln - Ll[t * PL + c]));
      }
      put(No, 2 * rt + ks, v);
    }
    if (quad == 0) ends[ch * DK + c] = __builtin_amdgcn_exp2f((float)Ln);
  }
  // M inside the block: lane (key c16, DK / 4 channels), its keys times the running product of the decays behind them
  constexpr int NC = DK / 4;
  float dg[16];
  {
    const int c0 = NC * quad, j = 16 * w + c16;
    float ke[NC];
#pragma unroll
    for (int u = 0; u < NC / 8; ++u) acts8(Kl, j, c0 + 8 * u, ke + 8 * u);
    float own = 0.f;  // the token's own term
    {
      float q[8];
#pragma unroll
      for (int u = 0; u < NC / 8; ++u) {
        acts8(Ql, j, c0 + 8 * u, q);
#pragma unroll
        for (int i = 0; i < 8; ++i) own += q[i] * ke[8 * u + i] * (BONUS ? bonus[(long)h * DK + c0 + 8 * u + i] : 1.f);
      }
      own = xor32_sum_f(xor16_sum(own));
    }
    // query j + d for d = 1 .. 15 (past the block's end: clamped, not stored).  Plain: the decays behind key j up to the
    // query's own; bonus: up to the token before it.  The rows of the next d are read ahead of this one's products.
    f32x4 gn[NC / 4], gv[NC / 4];
    u32x4 qn[NC / 8], qv[NC / 8];
    auto next = [&](int d) {
      const int t = min(j + d, 16 * w + 15), tg = BONUS ? min(j + d - 1, 16 * w + 15) : t;
#pragma unroll
      for (int u = 0; u < NC / 4; ++u) gn[u] = *reinterpret_cast<const f32x4*>(&Gl[tg * PG + c0 + 4 * u]);
#pragma unroll
      for (int u = 0; u < NC / 8; ++u) qn[u] = *reinterpret_cast<const u32x4*>(&Ql[t * PK + c0 + 8 * u]);
    };
    next(1);
    dg[0] = q_scale * own;
#pragma unroll
    for (int d = 1; d < 16; ++d) {
#pragma unroll
      for (int u = 0; u < NC / 4; ++u) gv[u] = gn[u];
#pragma unroll
      for (int u = 0; u < NC / 8; ++u) qv[u] = qn[u];
      if (d < 15) next(d + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (!BONUS || d > 1) {
#pragma unroll
        for (int u = 0; u < NC; ++u) ke[u] *= gv[u / 4][u & 3];
      }
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int u = 0; u < NC; u += 2) {
        const uint32_t x = qv[u / 8][(u & 7) >> 1];
        s0 += __builtin_bit_cast(float, x << 16) * ke[u];
        s1 += __builtin_bit_cast(float, x & 0xffff0000u) * ke[u + 1];
      }
      dg[d] = q_scale * xor32_sum_f(xor16_sum(s0 + s1));
    }
  }
  __syncthreads();  // L has been read
  float* M = KS == 1 ? Mx : Ml;
#pragma unroll
  for (int kt = 0; kt < 3; ++kt)
    if (kt < w) *reinterpret_cast<float4*>(&M[qi * PM + 16 * kt + 4 * quad]) = make_float4(p[kt][0], p[kt][1], p[kt][2], p[kt][3]);
#pragma unroll
  for (int d = 0; d < 16; ++d)  // query c16 + d of the block; its later keys are left out when M is read
    if ((d >> 2) == quad && c16 + d < 16) M[(16 * w + c16 + d) * PM + 16 * w + c16] = dg[d];
  __syncthreads();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    if (32 * ks > 16 * w + 15) continue;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = 32 * ks + 8 * quad + i;
      v[i] = j <= qi && j < n ? M[qi * PM + j] : 0.f;
    }
    put(Mo, 2 * w + ks, v);
  }
}

// MODE kWhole: workgroups own whole segments.  Else a segment is cut into spans of `span` chunks that run side by side: kSpanEnds
// leaves the end state of every span but a segment's last from a zero state in spans_s [span][head][dv][channels], its decays'
// products in spans_d [span][head][channels], and the state that the segment starts from in its last span's place; kSpanRun
// folds those in front of its own span, S <- diag(d_j) S + E_j.
template <int KS, int NT, int MODE>
__global__ __launch_bounds__(512, 2) void decay_chunk_scan_kernel(float* __restrict__ o, const bf16_t* __restrict__ qkv,
                                                                  long stride, int v_col, const float* __restrict__ mats,
                                                                  const float* __restrict__ ends, float* __restrict__ state,
                                                                  const int* __restrict__ cu, const int* __restrict__ ctx,
                                                                  const int* __restrict__ slot, int S_, int H, int dv, int span, int n_span,
                                                                  float* __restrict__ spans_s, float* __restrict__ spans_d) {
  constexpr int DK = 32 * KS, PK = DK + 8, NV = 16 * NT, PV = NV + 8, RTW = (2 * KS + 3) / 4;
  __shared__ __attribute__((aligned(16))) bf16_t Sl[2][3][NV * PK];  // the state before a chunk, [column][channel]
  __shared__ __attribute__((aligned(16))) bf16_t Vl[2][kChunk * PV];
  __shared__ __attribute__((aligned(16))) int first[2][NV];  // chunk_seg.h: rows from which a column is no number
  const int nz = dv / NV, pair = (blockIdx.x & 7) + 8 * (blockIdx.x / (8 * nz)), zb = (blockIdx.x >> 3) % nz;
  if (pair >= (MODE == kWhole ? S_ : n_span) * H) return;
  const int h = pair % H, dvb = zb * NV, sp_i = n_span - 1 - pair / H;
  ChunkAt at = {0, 0, 0, 0, 1};
  SegAt own;
  if (MODE == kWhole) {
    own = segment_in_turn(cu, slot, S_, pair / H, H * nz);
    at.seg = own.seg;
  } else {
    at = chunk_at(cu, S_, sp_i, span * kChunk);
    if (at.seg < 0) return;
    own = {at.seg, slot[at.seg], at.row, at.row + at.n};
    if (MODE == kSpanEnds && (at.k == at.count - 1 || own.slot < 0)) return;
  }
  const int s = own.seg, sl = own.slot, t0 = own.t0, t1 = own.t1;
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3;
  const bool outs = wave < 4;  // wave-uniform
  const long inner = (long)H * dv;
  if (sl < 0) {  // padding rows: defined output, no state
    for (int i = tid; i < (t1 - t0) * NV; i += 512) o[(long)(t0 + i / NV) * inner + (long)h * dv + dvb + (i % NV)] = 0.f;
    return;
  }
  if (t1 <= t0) return;
  const int c0 = first_chunk(cu, s) + (MODE == kWhole ? 0 : at.k * span);
  f32x4 S[RTW][NT];  // S[16 (w RTW + r) + 4 quad + i][16 ct + c16]
  float* sp = state + (((long)sl * H + h) * dv + dvb) * DK;
  const bool carried = ctx[s] > 0 && (MODE == kWhole || at.count == 1 || (MODE == kSpanEnds && at.k == 0)), mine = !outs && w * RTW < 2 * KS;
#pragma unroll
  for (int r = 0; r < RTW; ++r)
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      S[r][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int row = 16 * (w * RTW + r) + 4 * quad;
      if (carried && mine && row < DK) {
        const float4 v = *reinterpret_cast<const float4*>(sp + (long)(16 * ct + c16) * DK + row);
        S[r][ct] = f32x4{v.x, v.y, v.z, v.w};
      }
    }
  // the place of span j of this segment; this thread's part of a state there
  auto end_of = [&](int j) { return spans_s + (((long)(sp_i - at.k + j) * H + h) * dv + dvb) * DK; };
  auto each = [&](auto f) {
#pragma unroll
    for (int r = 0; r < RTW; ++r)
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        const int row = 16 * (w * RTW + r) + 4 * quad;
        if (mine && row < DK) f(S[r][ct], (long)(16 * ct + c16) * DK + row, r, row);
      }
  };
  float4 prod[RTW];
#pragma unroll
  for (int r = 0; r < RTW; ++r) prod[r] = make_float4(1.f, 1.f, 1.f, 1.f);
  if (MODE == kSpanEnds && at.k == 0) {
    float* p = end_of(at.count - 1);
    each([&](f32x4& v, long o, int, int) {
      *reinterpret_cast<f32x4*>(p + o) = v;
      v = f32x4{0.f, 0.f, 0.f, 0.f};
    });
  }
  if (MODE == kSpanRun && at.count > 1) {
    const float* p = end_of(at.count - 1);
    each([&](f32x4& v, long o, int, int) { v = *reinterpret_cast<const f32x4*>(p + o); });
    for (int j = 0; j < at.k; ++j) {
      const float* e = end_of(j);
      const float* d = spans_d + ((long)(sp_i - at.k + j) * H + h) * DK;
      each([&](f32x4& v, long o, int, int row) {
        v = v * *reinterpret_cast<const f32x4*>(d + row) + *reinterpret_cast<const f32x4*>(e + o);
      });
    }
  }
  auto publish = [&](int buf) {
    if (MODE == kSpanEnds) return;  // nobody reads it
#pragma unroll
    for (int r = 0; r < RTW; ++r) {
      const int rt = w * RTW + r;
      if (mine && rt < 2 * KS) {
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {
          float x[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = S[r][ct][i];
          uint32_t p[3][2];
          split_pairs<2>(x, p[0], p[1], p[2]);
#pragma unroll
          for (int k = 0; k < 3; ++k)
            *reinterpret_cast<uint2*>(&Sl[buf][k][(16 * ct + c16) * PK + 16 * rt + 4 * quad]) = make_uint2(p[k][0], p[k][1]);
        }
      }
    }
  };
  // operands, fetched one chunk ahead as fp32 and split when their chunk begins: outs: fragments of Q' (KS) and M (2); else
  // N (2 RTW) and the ends of its rows
  constexpr int NF = KS + 2 > 2 * RTW ? KS + 2 : 2 * RTW;
  bf16x8 mf[3 * NF];
  f32x4 mn[2 * NF];
  float4 ef[RTW], en[RTW];
  constexpr int VW = NV * 64 / 512;  // values a thread stages: 2 NT
  uint32_t rv[VW / 2];
  const int vr = tid / (NV / VW), vc = VW * (tid % (NV / VW));
  auto fetch = [&](int tb) {
    const long ch = (long)(c0 + (tb - t0) / kChunk) * H + h;
    const float* m = mats + ch * kc_mats(DK) + lane * 4;
    if (outs) {
      if (MODE == kSpanEnds) return;
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) mn[i] = *reinterpret_cast<const f32x4*>(m + (long)(2 * KS * w + i) * 256);
      m += 64 * DK;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < 2 || w >= 2) mn[2 * KS + i] = *reinterpret_cast<const f32x4*>(m + (long)(4 * w + i) * 256);
    } else if (mine) {
      m += 64 * DK + 64 * 64;
#pragma unroll
      for (int i = 0; i < 4 * RTW; ++i) mn[i] = *reinterpret_cast<const f32x4*>(m + (long)min(4 * w * RTW + i, 8 * KS - 1) * 256);
#pragma unroll
      for (int r = 0; r < RTW; ++r)
        en[r] = *reinterpret_cast<const float4*>(ends + ch * DK + min(16 * (w * RTW + r) + 4 * quad, DK - 4));
    }
  };
  auto split = [&](auto frags) {
#pragma unroll
    for (int i = 0; i < decltype(frags)::value; ++i) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = mn[2 * i + (e >> 2)][e & 3];
      uint32_t x[3][4];
      split_pairs<4>(v, x[0], x[1], x[2]);
#pragma unroll
      for (int k = 0; k < 3; ++k) mf[3 * i + k] = frag(x[k]);
    }
  };
  auto fetch_v = [&](int tb) {
    const bf16_t* v = qkv + (long)(tb + min(vr, min(kChunk, t1 - tb) - 1)) * stride + v_col + (long)h * dv + dvb + vc;
    if constexpr (VW == 2) {
      rv[0] = *reinterpret_cast<const uint32_t*>(v);
    } else if constexpr (VW == 4) {
      const uint2 t = *reinterpret_cast<const uint2*>(v);
      rv[0] = t.x, rv[1] = t.y;
    } else {
      const uint4 t = *reinterpret_cast<const uint4*>(v);
      rv[0] = t.x, rv[1] = t.y, rv[2] = t.z, rv[3] = t.w;
    }
  };
  auto stage_v = [&](int buf, int n) {
    keep_finite<VW>(rv, vr, n, first[buf] + vc);
#pragma unroll
    for (int i = 0; i < VW / 2; ++i) *reinterpret_cast<uint32_t*>(&Vl[buf][vr * PV + vc + 2 * i]) = rv[i];
  };
  fetch_v(t0);
  fetch(t0);
  if (tid < 2 * NV) first[tid / NV][tid % NV] = kNone;
  lds_barrier();
  publish(0);
  stage_v(0, min(kChunk, t1 - t0));
  if (t0 + kChunk < t1) fetch_v(t0 + kChunk);
  int buf = 0;
  for (int tb = t0; tb < t1; tb += kChunk, buf ^= 1) {
    const int n = min(kChunk, t1 - tb);
    if (!outs) split(std::integral_constant<int, 2 * RTW>{});
    else if (MODE != kSpanEnds) split(std::integral_constant<int, KS + 2>{});
#pragma unroll
    for (int r = 0; r < RTW; ++r) ef[r] = en[r];
    if (tb + kChunk < t1) fetch(tb + kChunk);
    lds_barrier();  // this chunk's state and values are written; the other buffers have been read
    if (tb + kChunk < t1) {
      stage_v(buf ^ 1, min(kChunk, t1 - tb - kChunk));
      if (tb + 2 * kChunk < t1) fetch_v(tb + 2 * kChunk);
    }
    if (outs) {
      if (MODE != kSpanEnds && 16 * w < n) {
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {  // (column 16 ct + 4 quad + i, query c16)
          f32x4 d[3] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int k = 2; k >= 0; --k) {
              const bf16x8 x = *reinterpret_cast<const bf16x8*>(&Sl[buf][k][(16 * ct + c16) * PK + 32 * ks + 8 * quad]);
#pragma unroll
              for (int m = 2 - k; m >= 0; --m) d[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, mf[3 * ks + m], d[m], 0, 0, 0);
            }
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            if (ks == 1 && w < 2) continue;  // M is lower triangular
            const bf16x8 x = frag_down(Vl[buf], PV, 32 * ks + 8 * quad, 32 * ks + 8 * quad + 4, 16 * ct);
#pragma unroll
            for (int m = 2; m >= 0; --m) d[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, mf[3 * KS + 3 * ks + m], d[m], 0, 0, 0);
          }
          const int4 f = *reinterpret_cast<const int4*>(&first[buf][16 * ct + 4 * quad]);
          const int q = 16 * w + c16;
          if (q < n)
            *reinterpret_cast<float4*>(o + (long)(tb + q) * inner + (long)h * dv + dvb + 16 * ct + 4 * quad) =
                make_float4(q < f.x ? (d[2][0] + d[1][0]) + d[0][0] : NAN, q < f.y ? (d[2][1] + d[1][1]) + d[0][1] : NAN,
                            q < f.z ? (d[2][2] + d[1][2]) + d[0][2] : NAN, q < f.w ? (d[2][3] + d[1][3]) + d[0][3] : NAN);
        }
      }
    } else if (mine) {
      if (MODE == kSpanEnds)
#pragma unroll
        for (int r = 0; r < RTW; ++r)
          prod[r] = make_float4(prod[r].x * ef[r].x, prod[r].y * ef[r].y, prod[r].z * ef[r].z, prod[r].w * ef[r].w);
#pragma unroll
      for (int r = 0; r < RTW; ++r)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {
          S[r][ct][0] *= ef[r].x;
          S[r][ct][1] *= ef[r].y;
          S[r][ct][2] *= ef[r].z;
          S[r][ct][3] *= ef[r].w;
        }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {
          const bf16x8 x = frag_down(Vl[buf], PV, 32 * ks + 8 * quad, 32 * ks + 8 * quad + 4, 16 * ct);
#pragma unroll
          for (int m = 2; m >= 0; --m)
#pragma unroll
            for (int r = 0; r < RTW; ++r)
              S[r][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf[6 * r + 3 * ks + m], x, S[r][ct], 0, 0, 0);
        }
#pragma unroll
      for (int ct = 0; ct < NT; ++ct)
        if (first[buf][16 * ct + c16] < kNone) {
#pragma unroll
          for (int r = 0; r < RTW; ++r) S[r][ct] = f32x4{NAN, NAN, NAN, NAN};
        }
      publish(buf ^ 1);
    }
  }
  if (MODE == kSpanEnds) {
    sp = end_of(at.k);
    if (zb == 0 && c16 == 0) {
      float* d = spans_d + ((long)sp_i * H + h) * DK;
#pragma unroll
      for (int r = 0; r < RTW; ++r) {
        const int row = 16 * (w * RTW + r) + 4 * quad;
        if (mine && row < DK) *reinterpret_cast<float4*>(d + row) = prod[r];
      }
    }
  }
  if (MODE != kSpanRun || at.k == at.count - 1)
    each([&](f32x4& v, long o, int, int) { *reinterpret_cast<f32x4*>(sp + o) = v; });
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

// Chunks per span of a step cut into spans, 0: whole segments.  Cut where long chains leave the chip idle - spans then take 64 columns
// at once, a quarter of the operand traffic, and twice the state's products (us, whole / spans, 32 heads of 64 x 64: 1 x 8000 rows
// 420 / 259, 1 x 2048 86 / 72, 2 x 4000 305 / 259, 4 x 2048, not cut, 241 / 244; 16 heads 1 x 8000 242 / 133; plain, 16 heads of
// 128 x 128, 1 x 8000 599 / 451) - about 256 workgroups of them.
static int span_chunks(long T, int S, int longest, int H, int dv, int mode) {
  const long n = longest > 0 ? longest : S > 0 ? T / S : 0;
  const int cols = dv % 64 == 0 ? dv / 64 : dv % 32 == 0 ? dv / 32 : dv / 16;
  if (n <= 0 || mode == 1 || (mode == 0 && (n < 1536 || H * ((T + n - 1) / n) * (dv / 16) > 256))) return 0;
  const long want = T / kChunk * H * cols / 256;
  return (int)(want < 4 ? 4 : want > 32 ? 32 : want);
}

// bytes of workspace for T rows in S segments, the longest of `longest` rows (0: not known, the mean is taken); 0: not a case for
// these kernels (dk a multiple of 32 up to 128, dv of 16).  mode 1 / 2: whole segments / spans whatever the sizes
long k8sllm_hy_decay_chunk_ws(long T, int S, int longest, int H, int dk, int dv, int mode) {
  if (dk % 32 || dk < 32 || dk > 128 || dv % 16 || dv < 16) return 0;
  const int span = span_chunks(T, S, longest, H, dv, mode);
  return (T / kChunk + S) * H * (kc_mats(dk) + dk) * 4 + (span > 0 ? (T / (span * kChunk) + S) * H * (long)dk * (dv + 1) * 4 : 0);
}

// as k8sllm_hy_decay_scan's plain form (bonus nullptr) or bonus form, without unit norms
int k8sllm_hy_decay_chunk(float* o, const void* qkv, long stride, int q_col, int k_col, int v_col, const void* z, long z_stride,
                          const float* z_bias, const float* a_log, float inv_tau, int dkind, const float* bonus, float* state,
                          const int* cu, const int* ctx, const int* slot, int S, int H, int Gk, int dk, int dv, float q_scale,
                          void* ws, long T, int longest, int mode, hipStream_t s) {
  if (S <= 0 || T <= 0) return 0;
  if (k8sllm_hy_decay_chunk_ws(T, S, longest, H, dk, dv, mode) == 0 || Gk < 1 || H % Gk || dkind < 0 || dkind > 2 || (dkind == 0 && a_log == nullptr))
    return -1;
  const long nch = T / kChunk + S;
  float* mats = (float*)ws;
  float* ends = mats + nch * H * kc_mats(dk);
  const long pairs = (long)S * H;
  // narrow column blocks until they fill the chip: the chain of chunks bounds a block
  const int span = span_chunks(T, S, longest, H, dv, mode);
  const long n_span = span > 0 ? T / (span * kChunk) + S : S, units = n_span * H;
  float* spans_s = ends + nch * H * dk;
  float* spans_d = spans_s + units * dk * dv;
  const int nt = dv % 64 == 0 && (span > 0 || pairs * (dv / 16) >= 1024) ? 4 : dv % 32 == 0 && (span > 0 || pairs * (dv / 16) >= 512) ? 2 : 1;
  const dim3 grid((unsigned)((units + 7) / 8 * 8 * (dv / (16 * nt)))), pgrid((unsigned)nch, (unsigned)H);
#define K8SLLM_KCP(KS, B)                                                                                                    \
  hipLaunchKernelGGL((decay_chunk_prep_kernel<KS, B>), pgrid, dim3(256), 0, s, mats, ends, (const bf16_t*)qkv, stride, q_col, \
                     k_col, (const bf16_t*)z, z_stride, z_bias, a_log, inv_tau, dkind, bonus, cu, slot, S, H, Gk, q_scale)
#define K8SLLM_KCM(KS, NT, MODE)                                                                                             \
  hipLaunchKernelGGL((decay_chunk_scan_kernel<KS, NT, MODE>), grid, dim3(512), 0, s, o, (const bf16_t*)qkv, stride, v_col, mats, \
                     ends, state, cu, ctx, slot, S, H, dv, span, (int)n_span, spans_s, spans_d)
#define K8SLLM_KCS(KS, NT)                       \
  do {                                           \
    if (span > 0) {                              \
      K8SLLM_KCM(KS, NT, kSpanEnds);             \
      K8SLLM_KCM(KS, NT, kSpanRun);              \
    } else {                                     \
      K8SLLM_KCM(KS, NT, kWhole);                \
    }                                            \
  } while (0)
#define K8SLLM_KC(KS)                        \
  if (bonus != nullptr) K8SLLM_KCP(KS, true); \
  else K8SLLM_KCP(KS, false);                \
  if (nt == 4) K8SLLM_KCS(KS, 4);            \
  else if (nt == 2) K8SLLM_KCS(KS, 2);       \
  else K8SLLM_KCS(KS, 1)
  switch (dk / 32) {
    case 1: K8SLLM_KC(1); break;
    case 2: K8SLLM_KC(2); break;
    case 3: K8SLLM_KC(3); break;
    default: K8SLLM_KC(4); break;
  }
#undef K8SLLM_KC
#undef K8SLLM_KCM
#undef K8SLLM_KCS
#undef K8SLLM_KCP
  return (int)hipGetLastError();
}
}
