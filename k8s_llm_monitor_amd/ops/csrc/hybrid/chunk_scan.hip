// Linear attention with a fixed decay per head on the matrix cores (bf16 activations, prompts):
//
//   S_t = lam S_(t-1) + k_t v_t^T,   o_t = S_t^T q_t        (per head; S is [dk][dv], fp32)
//
// over chunks of 64 tokens: with i, j the places of a query and a key inside a chunk of n tokens,
//
//   o_i   = lam^(i+1) (q_i S_prev) + sum_(j <= i) lam^(i-j) (q_i . k_j) v_j
//   S_new = lam^n S_prev           + sum_j k_j (lam^(n-1-j) v_j)^T
//
// so only the state crosses chunks.  Every product has one operand of bf16 activations (q, k, v as they are) and runs on
// v_mfma_f32_16x16x32_bf16; the other operand - weighted scores, state, decayed values - is fp32 and goes in as three
// bf16 parts that add up to it exactly (split_bf16.h), so scores, decays and state are never rounded below 32 bits.
//
// A workgroup of eight waves owns (segment, head, 16 NT value columns): value columns are independent, which gives the
// sequential chain of chunks its parallel axis.  Waves 0 .. 3 compute the outputs of 16 queries each, transposed
// (query on the lane); at the same time waves 4 .. 7 update the state, whose rows they hold in registers, a share of the key
// dims each.  Keys, values and the decayed values' three parts
// are row-major in LDS and read down the columns by the transposing LDS read; the state is republished there once per
// chunk as three bf16 parts, [column][key dim].  The next chunk's rows are fetched into registers while this chunk's
// products run.
// What bounds it: the chain of LDS round trips and two barriers per chunk, 1.7 us (16 columns) to 4.4 us (64) a chunk and workgroup.
// Its fragments are on their way before the first product that takes one, and no LDS read or prefetched row stands behind a
// branch or goes through scratch: with one wait for every read and product it was 3.2 to 5.4 us.
// Measured, bf16, 16 heads of 128 x 128: 5 of 1500 to 1637 rows 113 us (the sequential scan 314; before 138), 1 x 8000 rows 216 us (1068;
// before 402).  Error against 64 bits, 1600 rows: outputs 1.4e-7 (scan
// 2.2e-7), state 1.3e-7 (2.2e-7).
#include "chunk_seg.h"
#include "split_bf16.h"

namespace k8sllm {

constexpr int kCsChunk = kChunk;

template <int KS, int NT>  // key dim / 32, value columns / 16 per workgroup
__global__ __launch_bounds__(512, 2) void chunk_scan_kernel(float* __restrict__ y, const bf16_t* __restrict__ vkq,
                                                         const float* __restrict__ decay,
                                                         float* __restrict__ state, const int* __restrict__ cu,
                                                         const int* __restrict__ ctx, const int* __restrict__ slot, int S_,
                                                         int H, int dv) {
  constexpr int DK = 32 * KS, PK = DK + 8, NV = 16 * NT, PV = NV + 8;
  constexpr int RTW = (2 * KS + 3) / 4;  // state row tiles per wave
  constexpr int KU = (KS + 1) / 2;                // 16-byte pieces of the keys per thread when staging
  constexpr int VPT = 2 * NT;                     // value columns per thread
  __shared__ __attribute__((aligned(16))) bf16_t Kl[kCsChunk * PK];
  __shared__ __attribute__((aligned(16))) bf16_t Vl[4][kCsChunk * PV];  // values, then the decayed values' three parts
  __shared__ __attribute__((aligned(16))) bf16_t Sl[3][NV * PK];        // the state before the chunk, [column][key dim]
  __shared__ float lam[kCsChunk + 1];                                   // the decay's powers
  __shared__ __attribute__((aligned(16))) int first[NV];                // chunk_seg.h: rows from which a column is no number
  // workgroups go round the eight XCDs: all column blocks of a (segment, head) pair on one, whose L2 then serves their
  // common keys and queries
  const int nz = dv / NV, pair = (blockIdx.x & 7) + 8 * (blockIdx.x / (8 * nz)), zb = (blockIdx.x >> 3) % nz;
  if (pair >= S_ * H) return;
  const SegAt at = segment_in_turn(cu, slot, S_, pair / H, H * nz);
  const int s = at.seg, sl = at.slot, t0 = at.t0, t1 = at.t1, h = pair % H, dvb = zb * NV;
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3;
  const bool outs = wave < 4;  // wave-uniform: outputs, else state
  const long inner = (long)H * dv, C = inner + 2L * H * DK;
  if (sl < 0) {  // padding rows: defined output, no state
    for (int i = tid; i < (t1 - t0) * NV; i += 512) y[(long)(t0 + i / NV) * inner + (long)h * dv + dvb + (i % NV)] = 0.f;
    return;
  }
  if (t1 <= t0) return;
  const bf16_t* vcol = vkq + (long)h * dv + dvb;
  const bf16_t* kcol = vkq + inner + (long)h * DK;
  const bf16_t* qcol = kcol + (long)H * DK;
  if (tid < NV) first[tid] = kNone;
  if (tid <= kCsChunk) lam[tid] = tid == 0 ? 1.f : powf(decay[h], (float)tid);
  // state tile (r, ct): S[16 (w RTW + r) + 4 quad + i][16 ct + c16]
  f32x4 S[RTW][NT];
  float* sp = state + ((long)sl * H + h) * DK * dv + dvb;
  const bool carried = ctx[s] > 0;
#pragma unroll
  for (int r = 0; r < RTW; ++r)
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * (w * RTW + r) + 4 * quad + i;
        S[r][ct][i] = carried && !outs && row < DK ? sp[(long)row * dv + 16 * ct + c16] : 0.f;
      }
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // (an array of uint4 went through scratch or LDS behind its loads)
  u32x4 rk[KU];
  uint32_t rv[VPT / 2];
  bf16x8 qn[KS];
  const int vr = tid / (NV / VPT), vc = VPT * (tid % (NV / VPT));  // the value row and columns this thread stages
  auto fetch = [&](int tb, int n) {
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int idx = min(tid + 512 * u, kCsChunk * DK / 8 - 1), row = idx / (DK / 8), c8 = idx - row * (DK / 8);
      rk[u] = *reinterpret_cast<const u32x4*>(kcol + (long)(tb + min(row, n - 1)) * C + 8 * c8);
    }
    const bf16_t* v = vcol + (long)(tb + min(vr, n - 1)) * C + vc;
    if constexpr (VPT == 2) {
      rv[0] = *reinterpret_cast<const uint32_t*>(v);
    } else if constexpr (VPT == 4) {
      const uint2 t = *reinterpret_cast<const uint2*>(v);
      rv[0] = t.x, rv[1] = t.y;
    } else {
      const uint4 t = *reinterpret_cast<const uint4*>(v);
      rv[0] = t.x, rv[1] = t.y, rv[2] = t.z, rv[3] = t.w;
    }
    if (!outs) return;
    const bf16_t* q = qcol + (long)(tb + min(16 * w + c16, n - 1)) * C + 8 * quad;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qn[ks] = *reinterpret_cast<const bf16x8*>(q + 32 * ks);
  };
  fetch(t0, min(kCsChunk, t1 - t0));
  for (int tb = t0; tb < t1; tb += kCsChunk) {
    const int n = min(kCsChunk, t1 - tb);
    lds_barrier();  // the previous chunk's reads of Kl, Vl, Sl are done (and lam is written)
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int idx = tid + 512 * u, row = idx / (DK / 8), c8 = idx - row * (DK / 8);
      if (KS % 2 == 0 || idx < kCsChunk * DK / 8) *reinterpret_cast<u32x4*>(&Kl[row * PK + 8 * c8]) = rk[u];
    }
    {
      const float f = vr < n ? lam[n - 1 - vr] : 0.f;
      float x[VPT];
      uint32_t p[3][VPT / 2];
#pragma unroll
      for (int i = 0; i < VPT / 2; ++i) {
        x[2 * i] = __uint_as_float(rv[i] << 16) * f;
        x[2 * i + 1] = __uint_as_float(rv[i] & 0xffff0000u) * f;
      }
      split_pairs<VPT / 2>(x, p[0], p[1], p[2]);
      const int o = vr * PV + vc;
      auto put = [&](bf16_t* d, const uint32_t* x) {
        if constexpr (VPT == 2) *reinterpret_cast<uint32_t*>(d) = x[0];
        else if constexpr (VPT == 4) *reinterpret_cast<uint2*>(d) = make_uint2(x[0], x[1]);
        else *reinterpret_cast<uint4*>(d) = make_uint4(x[0], x[1], x[2], x[3]);
      };
      keep_finite<VPT>(rv, vr, n, first + vc);  // (the state takes its values as they are)
      put(&Vl[0][o], rv);
#pragma unroll
      for (int k = 0; k < 3; ++k) put(&Vl[k + 1][o], p[k]);
    }
#pragma unroll
    for (int r = 0; r < RTW; ++r) {
      const int rt = w * RTW + r;
      if (!outs && rt < 2 * KS) {
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
    bf16x8 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = qn[ks];
    lds_barrier();
    if (tb + kCsChunk < t1) {  // in flight during the products
      fetch(tb + kCsChunk, min(kCsChunk, t1 - tb - kCsChunk));
    }
    if (outs && 16 * w < n) {
      const int qi = 16 * w + c16;
      // o[ct][i]: query 16 w + c16, value column 16 ct + 4 quad + i; the three parts in chains of their own
      // (each block's fragments are on their way before its first product)
      f32x4 o[NT];
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        bf16x8 x[KS][3];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int k = 0; k < 3; ++k) x[ks][k] = *reinterpret_cast<const bf16x8*>(&Sl[k][(16 * ct + c16) * PK + 32 * ks + 8 * quad]);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 part[3] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int k = 0; k < 3; ++k) part[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[ks][k], qf[ks], part[k], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[ct][i] = (part[2][i] + part[1][i]) + part[0][i];
      }
      const float gq = lam[qi + 1];
#pragma unroll
      for (int ct = 0; ct < NT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[ct][i] *= gq;
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {  // pairs of 16-key tiles
        if (2 * kp <= w) {
          float p[8], decays[8];  // read for every key: a read behind a condition is a branch and a wait each
          bf16x8 a[2][KS], v[NT];
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
              a[u][ks] = *reinterpret_cast<const bf16x8*>(&Kl[(32 * kp + 16 * u + c16) * PK + 32 * ks + 8 * quad]);
#pragma unroll
          for (int i = 0; i < 8; ++i) decays[i] = lam[max(qi - (32 * kp + 16 * (i >> 2) + 4 * quad + (i & 3)), 0)];
#pragma unroll
          for (int ct = 0; ct < NT; ++ct) v[ct] = frag_down(Vl[0], PV, 32 * kp + 4 * quad, 32 * kp + 16 + 4 * quad, 16 * ct);
          __builtin_amdgcn_sched_barrier(0);
          f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int u = 0; u < 2; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][ks], qf[ks], acc[u], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 8; ++i) {  // acc[i / 4][i % 4]: key 32 kp + 16 (i / 4) + 4 quad + i % 4
            const int j = 32 * kp + 16 * (i >> 2) + 4 * quad + (i & 3);
            p[i] = j <= qi ? acc[i >> 2][i & 3] * decays[i] : 0.f;
          }
          uint32_t pw[3][4];
          split_pairs<4>(p, pw[0], pw[1], pw[2]);
#pragma unroll
          for (int k = 2; k >= 0; --k)
#pragma unroll
            for (int ct = 0; ct < NT; ++ct) o[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[ct], frag(pw[k]), o[ct], 0, 0, 0);
        }
      }
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        const int4 f = *reinterpret_cast<const int4*>(&first[16 * ct + 4 * quad]);
        if (qi >= f.x) o[ct][0] = NAN;
        if (qi >= f.y) o[ct][1] = NAN;
        if (qi >= f.z) o[ct][2] = NAN;
        if (qi >= f.w) o[ct][3] = NAN;
      }
      if (qi < n) {
        float* yr = y + (long)(tb + qi) * inner + (long)h * dv + dvb + 4 * quad;
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
          *reinterpret_cast<float4*>(yr + 16 * ct) = make_float4(o[ct][0], o[ct][1], o[ct][2], o[ct][3]);
      }
    }
    const float gn = lam[n];
#pragma unroll
    for (int r = 0; r < RTW; ++r)
#pragma unroll
      for (int ct = 0; ct < NT; ++ct)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[r][ct][i] *= gn;
    if (!outs && w * RTW < 2 * KS) {
#pragma unroll
      for (int tk = 0; tk < 2; ++tk) {
        if (32 * tk < n) {
          const int r0 = 32 * tk + 8 * quad;
          bf16x8 a[RTW];
#pragma unroll
          for (int r = 0; r < RTW; ++r) a[r] = frag_down(Kl, PK, r0, r0 + 4, 16 * min(w * RTW + r, 2 * KS - 1));
#pragma unroll
          for (int k = 2; k >= 0; --k) {
            bf16x8 b[NT];
#pragma unroll
            for (int ct = 0; ct < NT; ++ct) b[ct] = frag_down(Vl[k + 1], PV, r0, r0 + 4, 16 * ct);
#pragma unroll
            for (int ct = 0; ct < NT; ++ct)
#pragma unroll
              for (int r = 0; r < RTW; ++r) S[r][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r], b[ct], S[r][ct], 0, 0, 0);
          }
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RTW; ++r)
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * (w * RTW + r) + 4 * quad + i;
        if (!outs && row < DK) sp[(long)row * dv + 16 * ct + c16] = S[r][ct][i];
      }
}

}  // namespace k8sllm

using namespace k8sllm;

// vkq [T][H*dv | H*dk | H*dk] bf16 (values, keys, queries), state [slots][H][dk][dv] fp32, y [T][H*dv] fp32.  Returns 1
// (nothing launched) for sizes that are not this kernel's: dk a multiple of 32 up to 128, dv of 16, rows 16-byte
// aligned.  nt: value-column tiles per workgroup, 1, 2 or 4 (0: chosen here).
extern "C" int k8sllm_hy_chunk_scan(float* y, const void* vkq, const float* decay, float* state, const int* cu, const int* ctx,
                                    const int* slot, int S, long T, int longest, int H, int dk, int dv, int nt, hipStream_t s) {
  if (S <= 0) return 0;
  if (dk % 32 || dk < 32 || dk > 128 || dv % 16 || dv < 16 || H < 1) return 1;
  if (nt != 0 && nt != 1 && nt != 2 && nt != 4) return -1;
  if (nt > 1 && dv % (16 * nt)) return 1;
  // column blocks repeat the scores' products, and a CU holds one: the narrowest that give it no second one (us for 16 / 32 / 64 columns,
  // 128 x 128: 16 heads, 1 x 8000 rows 216 / 340 / 500; 2 x 4000 118 / 177 / 251; 3 x 2700 154 / 124 / 174; 4 x 2048 118 / 95 / 131; 5 of
  // 1500 to 1637 143 / 149 / 113; 16 x 500 125 / 100 / 76).  Segments count by the longest one's length (0: not known): short ones beside it
  // are a chunk or two each
  const long pairs = (longest > 0 ? min((long)S, (T + longest - 1) / longest) : S) * H;
  if (nt == 0)
    for (nt = 1; nt < 4 && dv % (32 * nt) == 0 && pairs * (dv / (16 * nt)) > 256;) nt *= 2;
  const dim3 grid((unsigned)(((long)S * H + 7) / 8 * 8 * (dv / (16 * nt))));
#define K8SLLM_CS(KS, NT)                                                                                           \
  hipLaunchKernelGGL((chunk_scan_kernel<KS, NT>), grid, dim3(512), 0, s, y, (const bf16_t*)vkq, decay, state, cu, ctx, \
                     slot, S, H, dv)
#define K8SLLM_CSN(KS)            \
  if (nt == 4) K8SLLM_CS(KS, 4);  \
  else if (nt == 2) K8SLLM_CS(KS, 2); \
  else K8SLLM_CS(KS, 1)
  switch (dk / 32) {
    case 1: K8SLLM_CSN(1); break;
    case 2: K8SLLM_CSN(2); break;
    case 3: K8SLLM_CSN(3); break;
    default: K8SLLM_CSN(4); break;
  }
#undef K8SLLM_CSN
#undef K8SLLM_CS
  return (int)hipGetLastError();
}
