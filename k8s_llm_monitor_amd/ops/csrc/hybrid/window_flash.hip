// Windowed grouped-query attention of large bf16 prompt steps: window_attn.hip's operator (pages, masks, sink, cap,
// kept first positions and head gate as its header says) for key sizes 64 / 128 and value sizes 64 / 128.
//
// What bounds it: the matrix cores and the softmax's exponentials, once keys and values come in cheaply.  The
// register kernel of window_attn.hip fetches every K / V^T fragment from global memory for 32 query rows of ONE
// head and does the softmax bookkeeping per 16 keys.  Here
//  * a workgroup of 8 waves takes 256 / HW query rows of HW query heads of one kv head (HW = 1, 2, 4 or 8, dividing
//    Hq / G); a wave owns 32 rows of one head.  Tiles of 64 keys (four pages) are copied to LDS by global_load_lds,
//    16 bytes a lane, straight from the pages, once for all 8 waves: a ring of four tiles, one barrier per tile, three
//    tiles in flight;
//  * S^T[key][query] = K Q^T and O^T[dim][query] += V^T P^T on v_mfma_f32_32x32x16_bf16, the query on the lane, so that
//    maxima, sums and rescaling are lane-local but for one v_permlane32_swap; the score accumulator becomes the PV
//    operand in place.  K rows are read in the order that swaps bits 2 and 3 of the token number: then a lane's 8
//    scores of a 16-key group are 8 CONSECUTIVE tokens and its V^T fragment is one 16-byte piece of a dim's row;
//  * both LDS images are swizzled by 16-byte pieces through the copies' source addresses (LDS itself is filled in
//    lane order): K piece ^ row, V piece ^ bit 3 of the dim, so that a read's 16 lanes touch 16 different bank quads;
//  * the running maximum moves only when a tile's exceeds it by 2^8: weights stay <= 256, exact in fp32 and in their
//    bf16 rounding; the accumulator is rescaled on such a jump only.  Tiles inside every row's range are not masked,
//    tiles outside all rows' are not visited, and a wave skips the tiles that none of its rows sees.  Where a wave's rows see a
//    tile in part, the 8-token pieces of V^T that none of them sees are read from zeros, and what lies behind the workgroup's last
//    token (the last page's unused end) is cleared in LDS: a masked weight of zero would not take away a NaN.
// Measured (us, 128-wide heads, register kernel -> this one): 4 x 2048 rows, 16 query heads on 4 kv heads, window 1024:
// 201 -> 88 (586 TFLOP/s); 2 x 2000 rows behind 2816 cached ones: 399 -> 148 (843 TFLOP/s); one prompt of 8000: 977 -> 272
// (962 TFLOP/s); the same in capped chunks of 1024: 122 -> 93 (three transcendental instructions per score bound it).  The zeros for
// pieces that are not seen and the cleared page end are 1 to 3 of these us.
#include "hy_common.h"

namespace k8sllm {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void gbl_void_t;

constexpr int kFlashRing = 4;
constexpr int kFlashIds = 4096;  // page ids that a workgroup keeps in LDS

// CAP 0: plain scores; 1: capped; 2: capped with a small cap and no sink, softmax without a running maximum
template <int DK, int DV, int HW, int CAP>
__global__ __launch_bounds__(512, 2) void window_flash_kernel(
    bf16_t* __restrict__ out, const bf16_t* __restrict__ qkv, long q_stride, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int* __restrict__ cu, const int* __restrict__ ctx,
    const int* __restrict__ block_tables, int bt_stride, int S, int Hq, int G, float scale, int window, int chunked,
    int keep, float cap, int sink, const float* __restrict__ sinks, const bf16_t* __restrict__ gate, long g_stride, int by_value) {
  constexpr int KS = DK / 16, DT = DV / 32, CHK = DK / 8;
  constexpr int WPH = 8 / HW, QR = 32 * WPH;
  constexpr int KB = 64 * DK * 2, TILE = KB + 64 * DV * 2;
  constexpr int NP = (DK + DV) / 64;  // 1 KiB copies per wave and tile
  constexpr int ZEROS = kFlashRing * TILE + kFlashIds * 4, ZB = (DT - 1) * 1024 + 16;
  __shared__ __attribute__((aligned(16))) char smem[ZEROS + ZB];
  int* s_blk = reinterpret_cast<int*>(smem + kFlashRing * TILE);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this workgroup's rows: q-blocks are numbered segment by segment, the last one first (most keys first)
  int seq = -1, qs = 0, L = 0, s0 = 0;
  {
    int total = 0;
    for (int b = 0; b < S; b += 64) {
      const int i = b + lane, n = i < S ? cu[i + 1] - cu[i] : 0;
      total += __builtin_amdgcn_readfirstlane((int)wave_sum_dpp((float)((n + QR - 1) / QR)));
    }
    int tile = total - 1 - (int)blockIdx.y;
    if (tile < 0) return;
    for (int b = 0; b < S && seq < 0; b += 64) {
      const int i = b + lane, c0 = i < S ? cu[i] : 0, n = i < S ? cu[i + 1] - c0 : 0, nt = (n + QR - 1) / QR;
      int incl = nt;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(incl, o, 64);
        if (lane >= o) incl += up;
      }
      const unsigned long long past = __ballot(incl > tile);
      if (past != 0) {
        const int f = __builtin_ctzll(past);
        seq = b + f;
        qs = (tile - (__shfl(incl, f, 64) - __shfl(nt, f, 64))) * QR;
        L = __shfl(n, f, 64);
        s0 = __shfl(c0, f, 64);
      } else {
        tile -= __shfl(incl, 63, 64);
      }
    }
    seq = __builtin_amdgcn_readfirstlane(seq);
    qs = __builtin_amdgcn_readfirstlane(qs);
    L = __builtin_amdgcn_readfirstlane(L);
    s0 = __builtin_amdgcn_readfirstlane(s0);
  }
  const int h = blockIdx.x * HW + wave / WPH, g = (blockIdx.x * HW) / (Hq / G);
  const int cst = ctx[seq];
  const int r32 = lane & 31, hh = lane >> 5;
  const int wq = qs + (wave % WPH) * 32;  // the wave's first row within the segment
  const bool any = wq < L;
  const int myq = wq + r32;
  const int my_p = cst + min(myq, L - 1), my_lo = first_key(my_p, window, chunked);
  const int pw0 = cst + min(wq, L - 1), pw1 = cst + min(wq + 31, L - 1);  // the wave's positions
  const int lo_w = first_key(pw0, window, chunked), lo_in = first_key(pw1, window, chunked);
  const int hi = cst + min(qs + QR, L);  // one past the workgroup's last position
  // tiles: those that hold kept keys, then from the first one that the workgroup's first row sees
  const int kt = (min(keep, hi) + 63) >> 6;
  const int w0 = max(kt, first_key(cst + qs, window, chunked) >> 6);
  const int nu = kt + max(0, ((hi - 1) >> 6) - w0 + 1);
  auto tile_of = [&](int u) { return u < kt ? u : w0 + u - kt; };

  const int* bt = block_tables + (long)seq * bt_stride;
  const int last_page = (hi - 1) >> 4;
  for (int i = tid; i < ZB / 4; i += 512) *reinterpret_cast<int*>(smem + ZEROS + 4 * i) = 0;
  for (int i = tid; i < nu * 4; i += 512) s_blk[i] = bt[min(4 * tile_of(i >> 2) + (i & 3), last_page)];
  bf16x8 qf[KS];
  {
    const bf16_t* qp = qkv + (long)(s0 + min(myq, L - 1)) * q_stride + (long)h * DK + 8 * hh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const bf16x8*>(qp + 16 * ks);
  }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(qf[ks]));  // the wait for these loads belongs before the copies
  __syncthreads();

  const long krs = (long)G * DK;
  // copy i of a wave: pieces of 1 KiB; K pieces hold 64 / CHK rows of one kv head, V pieces 32 dims of one page
  auto issue = [&](int u, int slot) {
    char* buf = smem + slot * TILE;
#pragma unroll
    for (int i = 0; i < DK / 64; ++i) {
      const int piece = wave * (DK / 64) + i;
      const int row = piece * (64 / CHK) + lane / CHK;
      const int ch = (lane % CHK) ^ (CHK == 16 ? (row & 15) : ((row >> 1) & 7));
      const long page = s_blk[4 * u + (piece * (64 / CHK) >> 4)];
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(k_cache + ((page << 4) + (row & 15)) * krs + (long)g * DK + ch * 8),
                                       (lds_void_t*)(buf + piece * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < DV / 64; ++i) {
      const int piece = wave * (DV / 64) + i;
      const int d = (piece % (DV / 32)) * 32 + (lane >> 1);
      const long page = s_blk[4 * u + piece / (DV / 32)];
      const int half = (lane & 1) ^ ((d >> 3) & 1);
      __builtin_amdgcn_global_load_lds((gbl_void_t*)(v_cache + ((page * G + g) * DV + d) * 16 + half * 8),
                                       (lds_void_t*)(buf + KB + piece * 1024), 16, 0, 0);
    }
  };

  constexpr float kLog2e = 1.44269504088896341f;
  const float sc2 = scale * kLog2e;
  const float cap2 = CAP ? cap * kLog2e : 0.f, icap = CAP ? scale / cap : 0.f;
  const float k1 = CAP ? icap * 2.f * kLog2e : 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m = sink ? (sinks != nullptr ? sinks[h] * kLog2e : 0.f) : -1e30f, l = sink && hh == 0 ? 1.f : 0.f;

  // token order of K rows: MFMA row i of a 16-row group reads the token with bits 2 and 3 swapped
  const int krow = (r32 & ~12) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);
  const int kswz = CHK == 16 ? (krow & 15) : ((krow >> 1) & 7);
  issue(0, 0);
  if (nu > 1) issue(1, 1);
  if (nu > 2) issue(2, 2);
  for (int u = 0; u < nu; ++u) {
    // this wave's pieces of tile u have landed; those of u + 1 and u + 2 may still fly
    if (u + 2 < nu) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NP) : "memory");
    else if (u + 1 < nu) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave's pieces of tile u are there, and tile u - 1 has been read
    if (u + 3 < nu) issue(u + 3, (u + 3) % kFlashRing);
    const int k0 = tile_of(u) * 64;
    if (k0 + 64 > hi) {  // workgroup-uniform: the last tile
      for (int i = tid; i < 8 * DV; i += 512) {  // pieces of 8 tokens: page i / (2 DV), dim, half
        const int d = (i >> 1) % DV, half = (i & 1) ^ ((d >> 3) & 1);
        uint4* p = reinterpret_cast<uint4*>(smem + (u % kFlashRing) * TILE + KB + 16 * i);
        const int j = k0 + 16 * (i / (2 * DV)) + 8 * half;
        if (j + 8 > hi) *p = tokens_below(*p, j, hi);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
    }
    if (!any || k0 > pw1 || (k0 + 63 < lo_w && k0 >= keep)) continue;
    const char* kb = smem + (u % kFlashRing) * TILE;
    int vo[2][2];  // this lane's V^T pieces of a page (dims r32, r32 + 32, ..)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        vo[i][s] = (u % kFlashRing) * TILE + KB + (2 * i + s) * (DV * 32) + (r32 * 2 + (hh ^ ((r32 >> 3) & 1))) * 16;
    if (k0 + 63 > pw1 || (k0 < lo_w && k0 + 63 >= keep)) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int t0 = k0 + 32 * i + 16 * s + 8 * hh;
          if (t0 > pw1 || (t0 + 7 < lo_w && t0 >= keep)) vo[i][s] = ZEROS;
        }
    }
    f32x16 sa[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) sa[i][r] = 0.f;
    {
      bf16x8 kf[KS][2];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          kf[ks][i] = *reinterpret_cast<const bf16x8*>(kb + (32 * i + krow) * (DK * 2) + (((2 * ks + hh) ^ kswz) << 4));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i) sa[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks][i], qf[ks], sa[i], 0, 0, 0);
    }
    // sa[i][8 s + j]: token k0 + 32 i + 16 s + 8 hh + j
    const bool inner = (k0 >= lo_in || k0 + 63 < keep) && k0 + 63 <= pw0;
    if (CAP == 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          sa[i][r] = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(sa[i][r] * k1));
    }
    const float mul = CAP ? 1.f : sc2;
    if (CAP != 2 && !inner) {
      const int base = k0 + 8 * hh, up = my_p - base, dn = my_lo - base, kp = keep - base;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = 32 * i + 16 * (r >> 3) + (r & 7);
          if (c > up || (c < dn && c >= kp)) sa[i][r] = -INFINITY;
        }
    }
    bf16x8 vf[2][2][DT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) vf[i][s][dt] = *reinterpret_cast<const bf16x8*>(smem + vo[i][s] + 1024 * dt);
    __builtin_amdgcn_sched_barrier(0);
    if (CAP != 2) {
      float mq[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        mq[c] = fmaxf(sa[c >> 1][8 * (c & 1)], sa[c >> 1][8 * (c & 1) + 1]);
#pragma unroll
        for (int r = 2; r < 8; ++r) mq[c] = fmaxf(mq[c], sa[c >> 1][8 * (c & 1) + r]);
      }
      const float mt = xor32_max_f(fmaxf(fmaxf(mq[0], mq[1]), fmaxf(mq[2], mq[3]))) * mul;
      const float mn = mt > m + 8.f ? mt : m;
      if (__builtin_amdgcn_ballot_w64(mn != m) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(m - mn);
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
        m = mn;
      }
    }
    float rq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x = sa[i][8 * s + j];
          if (CAP == 2)  // exp(cap tanh(score / cap)) in base 2
            p[j] = __builtin_amdgcn_exp2f(cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * k1)));
          else
            p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(x, mul, -m));
        }
        if (CAP == 2 && !inner) {
          const int base = k0 + 32 * i + 16 * s + 8 * hh, up = my_p - base, dn = my_lo - base, kp = keep - base;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (j > up || (j < dn && j >= kp)) p[j] = 0.f;
        }
        bf16x8 pb;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          rq[2 * i + s] += p[j];
          pb[j] = (__bf16)p[j];
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i][s][dt], pb, o[dt], 0, 0, 0);
      }
    l += (rq[0] + rq[1]) + (rq[2] + rq[3]);  // this lane's half of the keys; the halves meet at the end
  }
  l = xor32_sum_f(l);
  if (myq >= L) return;
  float inv = l > 0.f ? 1.f / l : 0.f;
  const bf16_t* gv = by_value ? gate + (long)(s0 + myq) * g_stride + (long)h * DV + 4 * hh : nullptr;
  if (gate != nullptr && !by_value) inv *= sigmoid_f(bf2f(gate[(long)(s0 + myq) * g_stride + h]));
  bf16_t* op = out + (long)(s0 + myq) * Hq * DV + (long)h * DV + 4 * hh;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint2 v;
      v.x = pack2(o[dt][4 * k] * inv, o[dt][4 * k + 1] * inv);
      v.y = pack2(o[dt][4 * k + 2] * inv, o[dt][4 * k + 3] * inv);
      if (by_value) v = gate_rounded(v, *reinterpret_cast<const uint2*>(gv + 32 * dt + 8 * k));
      *reinterpret_cast<uint2*>(op + 32 * dt + 8 * k) = v;
    }
}

}  // namespace k8sllm

using namespace k8sllm;

// 0: launched; 1: not a case for this kernel (the caller takes another one); else an error
extern "C" int k8sllm_hy_window_flash(void* out, const void* qkv, long q_stride, const void* k_cache, const void* v_cache,
                                      const int* cu, const int* ctx, const int* block_tables, int bt_stride, int S, long T,
                                      int Hq, int G, int dk, int dv, float scale, int window, int chunked, int keep, float cap,
                                      int plain_cap, int sink, const float* sinks, const void* gate, long g_stride, int by_value,
                                      hipStream_t s) {
  const int R = Hq / G;
  const int hw = R % 8 == 0 ? 8 : R % 4 == 0 ? 4 : R % 2 == 0 ? 2 : 1;
  const int qr = 256 / hw;
  if (!(scale > 0.f) || (dk != 64 && dk != 128) || (dv != 64 && dv != 128)) return 1;
  // page ids of a workgroup's tiles: all of a sequence's pages, or the window's and the kept tiles'
  const long ids = 4 * (((long)bt_stride + 3) / 4);
  const long near = window > 0 ? 4 * (((long)window + qr + 126) / 64 + ((long)keep + 63) / 64 + 1) : ids;
  if ((ids < near ? ids : near) > kFlashIds) return 1;
  const dim3 grid((unsigned)(Hq / hw), (unsigned)(T / qr + S));
#define K8SLLM_WF(DK, DV, HW, CAP)                                                                                     \
  hipLaunchKernelGGL((window_flash_kernel<DK, DV, HW, CAP>), grid, dim3(512), 0, s, (bf16_t*)out, (const bf16_t*)qkv,    \
                     q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, cu, ctx, block_tables, bt_stride, S, Hq, \
                     G, scale, window, chunked, keep, cap, sink, sinks, (const bf16_t*)gate, g_stride, by_value)
#define K8SLLM_WFC(DK, DV, HW)                        \
  if (cap > 0.f && plain_cap) K8SLLM_WF(DK, DV, HW, 2); \
  else if (cap > 0.f) K8SLLM_WF(DK, DV, HW, 1);       \
  else K8SLLM_WF(DK, DV, HW, 0)
#define K8SLLM_WFH(DK, DV)                  \
  if (hw == 8) { K8SLLM_WFC(DK, DV, 8); }   \
  else if (hw == 4) { K8SLLM_WFC(DK, DV, 4); } \
  else if (hw == 2) { K8SLLM_WFC(DK, DV, 2); } \
  else { K8SLLM_WFC(DK, DV, 1); }
  if (dk == 64 && dv == 64) { K8SLLM_WFH(64, 64); }
  else if (dk == 64) { K8SLLM_WFH(64, 128); }
  else if (dv == 64) { K8SLLM_WFH(128, 64); }
  else { K8SLLM_WFH(128, 128); }
#undef K8SLLM_WFH
#undef K8SLLM_WFC
#undef K8SLLM_WF
  return (int)hipGetLastError();
}
