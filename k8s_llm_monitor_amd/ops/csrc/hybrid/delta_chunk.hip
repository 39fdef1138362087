// The delta rule with one decay per head, bf16 prompts, in chunks of 64 tokens on the matrix cores.
//
//   S <- g_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t        (per head; S is [dk][dv], fp32)
//
// Inside a chunk of n tokens, with L_i the sum of log2 g up to token i, k and q already scaled to unit vectors:
//   A_ij = beta_i (k_i . k_j) 2^(L_i - L_j)  (j < i),   T = (1 + A)^-1,   W = T diag(beta),   P_ij = (q_i . k_j) 2^(L_i - L_j)  (j <= i)
//   R = V - diag(2^L) K S_prev                    (the rows that the chunk's updates start from)
//   O = diag(2^L) Q S_prev + M R                  M = P W
//   S = 2^L_n S_prev + N R                        N = K^T diag(2^(L_n - L)) W
// Nothing but R, O and S depends on the state, so two launches:
//  * delta_prep: a workgroup per (chunk, head), all of them in parallel: dot products on bf16 matrix instructions (exact
//    products of activations), the 64 x 64 triangular inverse by one wave (a column per lane, forward substitution in
//    registers), M and N; these are left in a workspace as three bf16 parts each, in operand order of the consumer, with the
//    row factors 2^L / |k|, 2^L / |q| and 2^L_n;
//  * delta_scan: a workgroup of eight waves per (segment, head, 16 NT value columns) walks the chunks; waves 0 .. 3 take
//    Q S and O, waves 4 .. 7 K S, R and S, 16 tokens each (then a share of the key dims).  K and Q are activations (exact
//    bf16, their scales are row factors), so S goes into those products as three bf16 parts (split_bf16.h); M R and N R
//    take the six products of two three-part operands that matter at 2^-24.  R and S pass between the waves through
//    LDS as three parts; all other operands are fetched straight into operand registers one chunk ahead.
// Sums of log2 g are kept in 64 bits: differences of large sums lose nothing.  Everything else is fp32.
// What bounds it: the chain K S -> R -> N R -> S per chunk, two barriers long, 1.3 us without its loads; the workspace's traffic (72 KiB
// per chunk and head, read by every column block, at dk 128), 0.8 us of a workgroup's load path.  Loads at the head of a chunk delayed its
// chain by all of that, branches around them made their first use wait for them: 2.5 us a chunk, 2.2 now.
// Measured, 16 heads of 128 x 128 on 8 key heads, both launches (us; the staged scan with its preparation): 1 x 8000 rows 362
// (1599), 4 x 2048 219 (544); 32 heads on 16, 4000 + 3000 + 1000 rows 472 (522 before).  Error against 64 bits at 4 x 2048: outputs 1.9e-7 (scan 3.0e-7),
// state 1.7e-7 (3.1e-7).
#include <type_traits>

#include "chunk_seg.h"
#include "split_bf16.h"

namespace k8sllm {

constexpr int kDcP = kChunk + 8;  // LDS pitch of [.][token] rows

// bf16 elements of M and N of one (chunk, head) in the workspace, and its floats (row factors, 2^L_n)
__host__ __device__ constexpr long dc_mats(int dk) { return 3L * 64 * (64 + dk); }
constexpr long kDcFac = 132;

template <int KS>
__global__ __launch_bounds__(256, 2) void delta_prep_kernel(bf16_t* __restrict__ mats, float* __restrict__ fac,
                                                            const bf16_t* __restrict__ qkv, long stride, int q_col, int k_col,
                                                            const bf16_t* __restrict__ z, long z_stride,
                                                            const float* __restrict__ z_bias, const float* __restrict__ a_log,
                                                            float inv_tau, int dkind, const bf16_t* __restrict__ beta,
                                                            long b_stride, const int* __restrict__ cu,
                                                            const int* __restrict__ slot, int S, int H, int Gk, float q_scale,
                                                            int unit) {
  constexpr int DK = 32 * KS, PK = DK + 8, PA = 68;
  __shared__ __attribute__((aligned(16))) bf16_t Kl[64 * PK];
  __shared__ __attribute__((aligned(16))) bf16_t Wl[3][64 * kDcP];  // W^T, later (2^(L_n - L) / |k| W)^T: [column][token]
  __shared__ __attribute__((aligned(16))) bf16_t Pl[3][64 * kDcP];  // first A as fp32 [64][PA], then P [query][token]
  __shared__ double Ll[64];
  __shared__ float nk[64], nq[64], bl[64];
  __shared__ int odd_row;  // the first token whose key, decay or beta is no number: M is NaN from there on (kNone: there is none)
  float* Al = reinterpret_cast<float*>(&Pl[0][0]);
  static_assert(64 * PA * 4 <= 3 * 64 * kDcP * 2, "A fits where P will be");
  const ChunkAt at = chunk_at(cu, S, blockIdx.x);
  if (at.seg < 0 || slot[at.seg] < 0) return;
  const int h = blockIdx.y, g = h / (H / Gk), n = at.n;
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, quad = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bf16_t* rows = qkv + (long)at.row * stride;
  const bf16_t* kb = rows + k_col + (long)g * DK;
  const bf16_t* qb = rows + q_col + (long)g * DK;
  // keys to LDS, squared lengths of keys and queries (four threads a row)
  {
    const int r = tid >> 2, c0 = (tid & 3) * (DK / 4);
    const bf16_t* kr = kb + (long)min(r, n - 1) * stride + c0;
    const bf16_t* qr = qb + (long)min(r, n - 1) * stride + c0;
    float sk = 0.f, sq = 0.f, odd = 0.f;  // odd: NaN if the key has an infinity or a NaN
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const uint4 kv = *reinterpret_cast<const uint4*>(kr + 8 * u), qv = *reinterpret_cast<const uint4*>(qr + 8 * u);
      *reinterpret_cast<uint4*>(&Kl[r * PK + c0 + 8 * u]) = kv;
      float a[8], b[8];
      unpack8(kv, a);
      unpack8(qv, b);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sk += a[i] * a[i];
        sq += b[i] * b[i];
        odd = fmaf(a[i], 0.f, odd);
      }
    }
    sk = lanes_sum<4>(sk);
    sq = lanes_sum<4>(sq);
    odd = lanes_sum<4>(odd);
    if ((tid & 3) == 0) {
      nk[r] = (unit ? 1.0f / sqrtf(sk + 1e-6f) : 1.f) + odd;
      nq[r] = unit ? q_scale / sqrtf(sq + 1e-6f) : q_scale;
    }
  }
  if (w == 0) {
    const long t = at.row + min(lane, n - 1);
    const float A = a_log != nullptr ? expf(a_log[h]) : 0.f;
    double L = lane < n ? (double)log2_decay(bf2f(z[t * z_stride + h]) + z_bias[h], dkind, A, inv_tau) : 0.0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double up = __shfl_up(L, o, 64);
      if (lane >= o) L += up;
    }
    Ll[lane] = L;
    bl[lane] = lane < n ? sigmoid_f(bf2f(beta[t * b_stride + h])) : 0.f;
  }
  __syncthreads();
  const int qi = 16 * w + c16;  // this lane's row of A and P
  const double Lq = Ll[qi];
  float p[4][4];
  {
    bf16x8 kf[KS], qf[KS];
    const bf16_t* qr = qb + (long)min(qi, n - 1) * stride + 8 * quad;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kf[ks] = *reinterpret_cast<const bf16x8*>(&Kl[qi * PK + 32 * ks + 8 * quad]);
      qf[ks] = *reinterpret_cast<const bf16x8*>(qr + 32 * ks);
    }
    const float ba = bl[qi] * nk[qi], bq = nq[qi];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f}, b = a;
      if (kt <= w) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8 r = *reinterpret_cast<const bf16x8*>(&Kl[(16 * kt + c16) * PK + 32 * ks + 8 * quad]);
          a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r, kf[ks], a, 0, 0, 0);
          b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(r, qf[ks], b, 0, 0, 0);
        }
      }
      float av[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {  // key 16 kt + 4 quad + i
        const int j = 16 * kt + 4 * quad + i;
        const float e = nk[j] * __builtin_amdgcn_exp2f((float)(Lq - Ll[j]));
        av[i] = j < qi ? a[i] * ba * e : 0.f;
        p[kt][i] = j <= qi ? b[i] * bq * e : 0.f;
      }
      *reinterpret_cast<float4*>(&Al[qi * PA + 16 * kt + 4 * quad]) = make_float4(av[0], av[1], av[2], av[3]);
    }
  }
  __syncthreads();
  float t[64];  // wave 0: column `lane` of T
  if (w == 0) {
    const float num = nk[lane] + (float)Ll[lane] + bl[lane];
    const unsigned long long odd = __ballot(lane < n && num != num);
    if (lane == 0) odd_row = odd != 0 ? (int)__builtin_ctzll(odd) : kNone;
    // A's rows come four values at a time, the same for every lane, twelve reads ahead of their products (one or two ahead the
    // wave spent three quarters of its time on the reads' latency)
    constexpr int AHEAD = 12;
    f32x4 ring[AHEAD];
    int li = 1, lj = 0, at_k = 0;
    auto load = [&](int k) {
      if (li < 64) ring[k % AHEAD] = *reinterpret_cast<const f32x4*>(&Al[li * PA + lj]);
      if ((lj += 4) >= li) ++li, lj = 0;
    };
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) load(k);
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      float s0 = lane == i ? 1.f : 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll
      for (int j = 0; j < i; j += 4) {
        const f32x4 a = ring[at_k % AHEAD];
        s0 -= a[0] * t[j];
        if (j + 1 < i) s1 -= a[1] * t[j + 1];
        if (j + 2 < i) s2 -= a[2] * t[j + 2];
        if (j + 3 < i) s3 -= a[3] * t[j + 3];
        load(at_k + AHEAD);
        ++at_k;
        __builtin_amdgcn_sched_barrier(0);
      }
      t[i] = (s0 + s1) + (s2 + s3);
    }
    const float b = bl[lane];
#pragma unroll
    for (int i = 0; i < 64; ++i) t[i] *= b;
#pragma unroll
    for (int i = 0; i < 64; i += 8) {
      uint32_t x[3][4];
      split_pairs<4>(t + i, x[0], x[1], x[2]);
#pragma unroll
      for (int k = 0; k < 3; ++k) *reinterpret_cast<uint4*>(&Wl[k][lane * kDcP + i]) = make_uint4(x[k][0], x[k][1], x[k][2], x[k][3]);
    }
    if (odd_row < kNone) {  // M's rows in front of that one do not see what it and its beta make of later ones and of its column
#pragma unroll 1
      for (int i = 0; i < 64; ++i)
        if (i >= odd_row || i < lane)
          for (int k = 0; k < 3; ++k) Wl[k][lane * kDcP + i] = 0;
    }
  }
  __syncthreads();  // A has been read
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) {
    uint32_t x[3][2];
    split_pairs<2>(p[kt], x[0], x[1], x[2]);
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<uint2*>(&Pl[k][qi * kDcP + 16 * kt + 4 * quad]) = make_uint2(x[k][0], x[k][1]);
  }
  const long ch = (long)blockIdx.x * H + h;
  bf16_t* Mo = mats + ch * dc_mats(DK);
  bf16_t* No = Mo + 3 * 64 * 64;
  const double Ln = Ll[63];
  if (tid < 64) {
    const float e = __builtin_amdgcn_exp2f((float)Ll[tid]);
    fac[ch * kDcFac + tid] = e * nq[tid];
    fac[ch * kDcFac + 64 + tid] = e * nk[tid];
    if (tid == 0) fac[ch * kDcFac + 128] = __builtin_amdgcn_exp2f((float)Ln);
  }
  __syncthreads();
  // transposed products: rows = columns j of M and N in the order that gives a lane 8 consecutive ones over two tiles
  auto wrow = [&](int ks, int a) { return 32 * ks + 8 * (c16 >> 2) + (c16 & 3) + 4 * a; };
  auto put = [&](bf16_t* o, int tile, const f32x4& lo, const f32x4& hi) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = lo[i], v[4 + i] = hi[i];
    uint32_t x[3][4];
    split_pairs<4>(v, x[0], x[1], x[2]);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      *reinterpret_cast<uint4*>(o + ((tile * 3 + k) * 64 + lane) * 8) = make_uint4(x[k][0], x[k][1], x[k][2], x[k][3]);
  };
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {  // M rows 16 w .., columns 32 ks ..
    if (32 * ks > 16 * w + 15) continue;
    f32x4 d[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int tk = 0; tk < 2; ++tk) {
      if (tk < ks || 32 * tk > 16 * w + 15) continue;
      bf16x8 b[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) b[k] = *reinterpret_cast<const bf16x8*>(&Pl[k][qi * kDcP + 32 * tk + 8 * quad]);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int k = 2; k >= 0; --k) {
          const bf16x8 x = *reinterpret_cast<const bf16x8*>(&Wl[k][wrow(ks, a) * kDcP + 32 * tk + 8 * quad]);
#pragma unroll
          for (int m = 2 - k; m >= 0; --m) d[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, b[m], d[a], 0, 0, 0);
        }
    }
    if (qi >= odd_row) d[0] = d[1] = f32x4{NAN, NAN, NAN, NAN};
    put(Mo, 2 * w + ks, d[0], d[1]);
  }
  __syncthreads();
  if (w == 0) {
#pragma unroll
    for (int i = 0; i < 64; i += 8) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = t[i + j] * (__builtin_amdgcn_exp2f((float)(Ln - Ll[i + j])) * nk[i + j]);
      uint32_t x[3][4];
      split_pairs<4>(v, x[0], x[1], x[2]);
#pragma unroll
      for (int k = 0; k < 3; ++k) *reinterpret_cast<uint4*>(&Wl[k][lane * kDcP + i]) = make_uint4(x[k][0], x[k][1], x[k][2], x[k][3]);
    }
  }
  __syncthreads();
  for (int rt = w; rt < 2 * KS; rt += 4) {  // N rows 16 rt ..
    bf16x8 b[2];
#pragma unroll
    for (int tk = 0; tk < 2; ++tk) b[tk] = frag_down(Kl, PK, 32 * tk + 8 * quad, 32 * tk + 8 * quad + 4, 16 * rt);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      f32x4 d[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int tk = 0; tk < 2; ++tk) {
          if (tk < ks) continue;  // W is lower triangular
#pragma unroll
          for (int k = 2; k >= 0; --k) {
            const bf16x8 x = *reinterpret_cast<const bf16x8*>(&Wl[k][wrow(ks, a) * kDcP + 32 * tk + 8 * quad]);
            d[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, b[tk], d[a], 0, 0, 0);
          }
        }
      put(No, 2 * rt + ks, d[0], d[1]);
    }
  }
}

template <int KS, int NT>
__global__ __launch_bounds__(512, 2) void delta_scan_kernel(float* __restrict__ o, const bf16_t* __restrict__ qkv, long stride,
                                                            int q_col, int k_col, int v_col, const bf16_t* __restrict__ mats,
                                                            const float* __restrict__ fac, float* __restrict__ state,
                                                            const int* __restrict__ cu, const int* __restrict__ ctx,
                                                            const int* __restrict__ slot, int S_, int H, int Gk, int dv) {
  constexpr int DK = 32 * KS, PK = DK + 8, NV = 16 * NT, RTW = (2 * KS + 3) / 4;
  __shared__ __attribute__((aligned(16))) bf16_t Sl[3][NV * PK];    // the state before the chunk, [column][key dim]
  __shared__ __attribute__((aligned(16))) bf16_t Rl[3][NV * kDcP];  // R, [column][token]
  __shared__ __attribute__((aligned(16))) int first[NV];            // chunk_seg.h: rows from which a column is no number
  // all column blocks of a (segment, head) pair on one XCD: its L2 then serves their common operands
  const int nz = dv / NV, pair = (blockIdx.x & 7) + 8 * (blockIdx.x / (8 * nz)), zb = (blockIdx.x >> 3) % nz;
  if (pair >= S_ * H) return;
  const SegAt at = segment_in_turn(cu, slot, S_, pair / H, H * nz);
  const int s = at.seg, sl = at.slot, t0 = at.t0, t1 = at.t1, h = pair % H, dvb = zb * NV, g = h / (H / Gk);
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3;
  const bool outs = wave < 4;  // wave-uniform
  const long inner = (long)H * dv;
  if (sl < 0) {  // padding rows: defined output, no state
    for (int i = tid; i < (t1 - t0) * NV; i += 512) o[(long)(t0 + i / NV) * inner + (long)h * dv + dvb + (i % NV)] = 0.f;
    return;
  }
  if (t1 <= t0) return;
  const int c0 = first_chunk(cu, s);
  // state tile (r, ct): S[16 (w RTW + r) + 4 quad + i][16 ct + c16]; the slot holds a column's key dims contiguous
  f32x4 S[RTW][NT];
  float* sp = state + (((long)sl * H + h) * dv + dvb) * DK;
  const bool carried = ctx[s] > 0, mine = !outs && w * RTW < 2 * KS;
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
  auto publish = [&]() {
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
            *reinterpret_cast<uint2*>(&Sl[k][(16 * ct + c16) * PK + 16 * rt + 4 * quad]) = make_uint2(p[k][0], p[k][1]);
        }
      }
    }
  };
  // operands of a chunk, fetched one chunk ahead (two sets in turn): this wave's 16 rows of Q or K, their row factors, M's tiles or
  // N's, the values that R starts from
  constexpr int NF = RTW > 1 ? 6 * RTW : 6;
  struct Operands {
    bf16x8 rows[KS], m[NF];
    float f[4], dl;  // outs: f[0] is this lane's query
    bf16_t v[4][NT];
  } ops[2];
  const bf16_t* rb = qkv + (outs ? q_col : k_col) + (long)g * DK + 8 * quad;
  // The same number of loads for every chunk and wave of a kind, with no branch around them (past the last chunk they repeat it): only
  // then does the use of one chunk's operands leave the next one's on their way.
  auto fetch = [&](auto queries, int tb, Operands& x) {
    tb = min(tb, t0 + (t1 - 1 - t0) / kChunk * kChunk);
    const int n = min(kChunk, t1 - tb);
    const long ch = (long)(c0 + (tb - t0) / kChunk) * H + h;
    const bf16_t* r = rb + (long)(tb + min(16 * w + c16, n - 1)) * stride;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) x.rows[ks] = *reinterpret_cast<const bf16x8*>(r + 32 * ks);
    const bf16_t* m = mats + ch * dc_mats(DK) + lane * 8;
    const float* f = fac + ch * kDcFac;
    if constexpr (decltype(queries)::value) {
#pragma unroll
      for (int i = 0; i < 6; ++i) x.m[i] = *reinterpret_cast<const bf16x8*>(m + (long)(6 * w + i) * 512);
      x.f[0] = f[16 * w + c16];
    } else {
      m += 3 * 64 * 64;
#pragma unroll
      for (int i = 0; i < 6 * RTW; ++i) x.m[i] = *reinterpret_cast<const bf16x8*>(m + (long)min(6 * w * RTW + i, 12 * KS - 1) * 512);
      x.dl = f[128];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x.f[i] = f[64 + 16 * w + 4 * quad + i];
        const bf16_t* v = qkv + (long)(tb + min(16 * w + 4 * quad + i, n - 1)) * stride + v_col + (long)h * dv + dvb + c16;
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) x.v[i][ct] = v[16 * ct];
      }
    }
  };
  publish();
  if (tid < NV) first[tid] = kNone;
  // three parts' products with this wave's rows; QUERIES: (S^T Q^T)[column 16 ct + 4 quad + i][query c16], else (K S)[token 4 quad +
  // i][column c16].  All of the state's fragments are on their way before the first product.
  auto dots = [&](auto queries, const bf16x8 (&rows)[KS], int ct) {
    bf16x8 x[KS][3];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int k = 0; k < 3; ++k) x[ks][k] = *reinterpret_cast<const bf16x8*>(&Sl[k][(16 * ct + c16) * PK + 32 * ks + 8 * quad]);
    f32x4 part[3] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}}, sum;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        part[k] = decltype(queries)::value ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[ks][k], rows[ks], part[k], 0, 0, 0)
                                           : __builtin_amdgcn_mfma_f32_16x16x32_bf16(rows[ks], x[ks][k], part[k], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] = (part[2][i] + part[1][i]) + part[0][i];
    return sum;
  };
  auto query_chunk = [&](int tb, const Operands& c, auto&& ahead) {
    const int n = min(kChunk, t1 - tb);
    f32x4 acc[NT];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) acc[ct] = dots(std::true_type{}, c.rows, ct);
    ahead();
    lds_barrier();  // Rl is written, Sl has been read
    if (16 * w >= n) return;
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      f32x4 d[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) d[0][i] = acc[ct][i] * c.f[0], d[1][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        if (ks == 1 && w < 2) continue;  // M is lower triangular
        bf16x8 x[3];
#pragma unroll
        for (int k = 2; k >= 0; --k) x[k] = *reinterpret_cast<const bf16x8*>(&Rl[k][(16 * ct + c16) * kDcP + 32 * ks + 8 * quad]);
#pragma unroll
        for (int k = 2; k >= 0; --k)
#pragma unroll
          for (int m = 2 - k; m >= 0; --m) d[m & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[k], c.m[3 * ks + m], d[m & 1], 0, 0, 0);
      }
      const int4 f = *reinterpret_cast<const int4*>(&first[16 * ct + 4 * quad]);
      const int q = 16 * w + c16;
      if (q < n)
        *reinterpret_cast<float4*>(o + (long)(tb + q) * inner + (long)h * dv + dvb + 16 * ct + 4 * quad) =
            make_float4(q < f.x ? d[0][0] + d[1][0] : NAN, q < f.y ? d[0][1] + d[1][1] : NAN, q < f.z ? d[0][2] + d[1][2] : NAN,
                        q < f.w ? d[0][3] + d[1][3] : NAN);
    }
  };
  auto key_chunk = [&](int tb, const Operands& c, auto&& ahead) {
    const int n = min(kChunk, t1 - tb);
    f32x4 acc[NT];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) acc[ct] = dots(std::false_type{}, c.rows, ct);
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = bf2f(c.v[i][ct]) - c.f[i] * acc[ct][i];
        if (!isfinite(x[i])) {
          const int row = 16 * w + 4 * quad + i;
          if (row < n) atomicMin(&first[16 * ct + c16], row);
          x[i] = 0.f;
        }
      }
      uint32_t p[3][2];
      split_pairs<2>(x, p[0], p[1], p[2]);
#pragma unroll
      for (int k = 0; k < 3; ++k)
        *reinterpret_cast<uint2*>(&Rl[k][(16 * ct + c16) * kDcP + 16 * w + 4 * quad]) = make_uint2(p[k][0], p[k][1]);
    }
    lds_barrier();  // Rl is written, Sl has been read
    if (!mine) return ahead();
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int r = 0; r < RTW; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[r][ct][i] *= c.dl;
    bf16x8 x[2][NT][3];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int ct = 0; ct < NT; ++ct)
#pragma unroll
        for (int k = 2; k >= 0; --k) x[ks][ct][k] = *reinterpret_cast<const bf16x8*>(&Rl[k][(16 * ct + c16) * kDcP + 32 * ks + 8 * quad]);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int ct = 0; ct < NT; ++ct)
#pragma unroll
        for (int k = 2; k >= 0; --k)
#pragma unroll
          for (int m = 2 - k; m >= 0; --m)
#pragma unroll
            for (int r = 0; r < RTW; ++r)
              S[r][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c.m[6 * r + 3 * ks + m], x[ks][ct][k], S[r][ct], 0, 0, 0);
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
      if (first[16 * ct + c16] < kNone) {
#pragma unroll
        for (int r = 0; r < RTW; ++r) S[r][ct] = f32x4{NAN, NAN, NAN, NAN};
      }
    publish();
    ahead();
  };
  // The two kinds of waves walk the chunks apart, meeting at two barriers each.  The next chunk's loads take a wave up to 0.8 us to
  // issue (104 KB a chunk and workgroup): the keys' waves do that when their state is published, the queries' behind their first products.
  auto walk = [&](auto queries, auto&& work) {
    auto chunk = [&](int tb, const Operands& c, Operands& next) {
      lds_barrier();  // Sl is written, Rl has been read
      work(tb, c, [&]() {
        __builtin_amdgcn_sched_barrier(0);
        fetch(queries, tb + kChunk, next);
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    fetch(queries, t0, ops[0]);
    for (int tb = t0; tb < t1; tb += 2 * kChunk) {
      chunk(tb, ops[0], ops[1]);
      if (tb + kChunk >= t1) break;
      chunk(tb + kChunk, ops[1], ops[0]);
    }
  };
  if (outs) walk(std::true_type{}, query_chunk);
  else walk(std::false_type{}, key_chunk);
  if (mine) {
#pragma unroll
    for (int r = 0; r < RTW; ++r)
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        const int row = 16 * (w * RTW + r) + 4 * quad;
        if (row < DK)
          *reinterpret_cast<float4*>(sp + (long)(16 * ct + c16) * DK + row) =
              make_float4(S[r][ct][0], S[r][ct][1], S[r][ct][2], S[r][ct][3]);
      }
  }
}

}  // namespace k8sllm

using namespace k8sllm;

extern "C" {

// bytes of workspace for T rows in S segments; 0: not a case for these kernels (dk a multiple of 32 up to 128, dv of 16)
long k8sllm_hy_delta_chunk_ws(long T, int S, int H, int dk, int dv) {
  if (dk % 32 || dk < 32 || dk > 128 || dv % 16 || dv < 16) return 0;
  return (T / kChunk + S) * H * (dc_mats(dk) * 2 + kDcFac * 4);
}

// o [T][H*dv] fp32; qkv rows with q, k ([Gk*dk]), v ([H*dv]) from q_col, k_col, v_col on, 16-byte aligned pieces; z, beta:
// column h of a row is head h's logit; state [slots][H][dv][dk] fp32
int k8sllm_hy_delta_chunk(float* o, const void* qkv, long stride, int q_col, int k_col, int v_col, const void* z, long z_stride,
                          const float* z_bias, const float* a_log, float inv_tau, int dkind, const void* beta, long b_stride,
                          float* state, const int* cu, const int* ctx, const int* slot, int S, int H, int Gk, int dk, int dv,
                          float q_scale, int unit, void* ws, long T, hipStream_t s) {
  if (S <= 0 || T <= 0) return 0;
  if (k8sllm_hy_delta_chunk_ws(T, S, H, dk, dv) == 0 || Gk < 1 || H % Gk || dkind < 0 || dkind > 2 || (dkind == 0 && a_log == nullptr))
    return -1;
  const long nch = T / kChunk + S;
  bf16_t* mats = (bf16_t*)ws;
  float* fac = (float*)(mats + nch * H * dc_mats(dk));
  // narrow column blocks until they fill the chip: the chain of chunks bounds a block
  const long pairs = (long)S * H;
  const int nt = dv % 32 == 0 && pairs * (dv / 16) >= 512 ? 2 : 1;
  const dim3 grid((unsigned)((pairs + 7) / 8 * 8 * (dv / (16 * nt))));
#define K8SLLM_DCS(KS, NT)                                                                                               \
  hipLaunchKernelGGL((delta_scan_kernel<KS, NT>), grid, dim3(512), 0, s, o, (const bf16_t*)qkv, stride, q_col, k_col, v_col, \
                     mats, fac, state, cu, ctx, slot, S, H, Gk, dv)
#define K8SLLM_DC(KS)                                                                                                       \
  hipLaunchKernelGGL((delta_prep_kernel<KS>), dim3((unsigned)nch, (unsigned)H), dim3(256), 0, s, mats, fac, (const bf16_t*)qkv, \
                     stride, q_col, k_col, (const bf16_t*)z, z_stride, z_bias, a_log, inv_tau, dkind, (const bf16_t*)beta,     \
                     b_stride, cu, slot, S, H, Gk, q_scale, unit);                                                            \
  if (nt == 2) K8SLLM_DCS(KS, 2);                                                                                           \
  else K8SLLM_DCS(KS, 1)
  switch (dk / 32) {
    case 1: K8SLLM_DC(1); break;
    case 2: K8SLLM_DC(2); break;
    case 3: K8SLLM_DC(3); break;
    default: K8SLLM_DC(4); break;
  }
#undef K8SLLM_DC
#undef K8SLLM_DCS
  return (int)hipGetLastError();
}
}
