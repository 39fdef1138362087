// Weight streams for a few rows: 16 output columns a wave, K in steps of 32, everything that v_mfma_f32_16x16x32_bf16 takes brought to
// LDS by global_load_lds, 16 bytes a lane, 1 KB (16 rows x 32 k) a piece.
// Why LDS and not registers: the instruction wants row lane % 16 in a lane, so a register load of row-major rows meets 16 cache lines in
// every 16 lanes and takes about 60 cycles of the load path (512 KB from L2 by one CU: 13 us, 3.6 us in lane order), and activations take as
// much of it as weights do.  A piece has four lanes a row; the chunk that lane l fetches is turned by the row, so that the
// fragments' reads (row lane % 16, chunk lane / 16) are spread over the banks.
#pragma once
#include <type_traits>

#include "hy_common.h"

namespace k8sllm {

// this lane's row and first k (of 32) in a piece, and where it finds its fragment in one
__device__ __forceinline__ int piece_row() { return (threadIdx.x & 63) >> 2; }
__device__ __forceinline__ int piece_k() { return 8 * ((threadIdx.x & 3) ^ ((threadIdx.x & 63) >> 4)); }
__device__ __forceinline__ int piece_frag() {
  const int lane = threadIdx.x & 63, c16 = lane & 15;
  return (4 * c16 + ((lane >> 4) ^ (c16 >> 2))) * 16;
}
__device__ __forceinline__ void load_piece(char* lds, const bf16_t* src) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) const void*)src, (__attribute__((address_space(3))) void*)lds, 16,
                                   0, 0);
}
template <int N>
__device__ __forceinline__ void loads_left() {  // waits until at most N of this wave's loads are on their way
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// NW waves of one workgroup share 16 MT rows, which come in chunks of 8 steps to a ring of two; each wave streams its own NS
// weight tiles through a private ring, 8 steps ahead.  Every output is one chain of products in the order of k.
template <int MT, int NS, int NW>
struct SharedRows {
  static constexpr int D = 8;  // steps of a chunk, and of the weights' ring
  static constexpr int SLOT = D * MT * 1024, RING = D * NS * 1024, BYTES = 2 * SLOT + NW * RING;
  static constexpr int PER = D * MT / NW;  // pieces of a chunk that a wave brings, all of one row tile
  static_assert(NW % MT == 0, "");

  // x(m): this lane's source in row tile m of the rows; w[t]: in weight tile t; nk: steps
  template <class X>
  static __device__ __forceinline__ void run(char* lds, X x, const bf16_t* const (&w)[NS], int nk, f32x4 (&acc)[MT][NS]) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rd = piece_frag();
    const int m0 = wave % MT, k0 = wave / MT;
    const bf16_t* xs = x(m0);
    char* ring = lds + 2 * SLOT + wave * RING;
    auto stage = [&](int c) {  // steps past the last repeat it; nothing multiplies them
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int ks = k0 + i * (NW / MT);
        load_piece(lds + (c & 1) * SLOT + (ks * MT + m0) * 1024, xs + 32 * min(c * D + ks, nk - 1));
      }
    };
    auto refill = [&](int d, int k) {
#pragma unroll
      for (int t = 0; t < NS; ++t) load_piece(ring + (d * NS + t) * 1024, w[t] + 32 * k);
    };
    auto chunk = [&](int c, auto whole) {
      constexpr bool WHOLE = decltype(whole)::value;  // every step, the next chunk and every refill are inside K
      if constexpr (WHOLE) loads_left<D * NS>();  // the chunk's pieces are older than the ring's
      else loads_left<0>();
      __builtin_amdgcn_s_barrier();  // every wave's pieces are there, and the other slot has been read
      if (WHOLE || (c + 1) * D < nk) stage(c + 1);
      auto step = [&](auto self, auto jc) {
        constexpr int j = decltype(jc)::value;
        if constexpr (j < D) {
          if (WHOLE || c * D + j < nk) {
            // younger than this step's weights: the D - 1 steps behind it and the chunk just begun
            if constexpr (WHOLE) loads_left<(D - 1) * NS + PER>();
            else if (j > 0) loads_left<0>();
            bf16x8 a[MT], b[NS];
#pragma unroll
            for (int t = 0; t < NS; ++t) b[t] = *reinterpret_cast<const bf16x8*>(ring + (j * NS + t) * 1024 + rd);
#pragma unroll
            for (int m = 0; m < MT; ++m) a[m] = *reinterpret_cast<const bf16x8*>(lds + (c & 1) * SLOT + (j * MT + m) * 1024 + rd);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (WHOLE || (c + 1) * D + j < nk) refill(j, (c + 1) * D + j);
#pragma unroll
            for (int t = 0; t < NS; ++t)
#pragma unroll
              for (int m = 0; m < MT; ++m) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b[t], acc[m][t], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          self(self, std::integral_constant<int, j + 1>{});
        }
      };
      step(step, std::integral_constant<int, 0>{});
    };
    stage(0);
#pragma unroll
    for (int d = 0; d < D; ++d) refill(d, min(d, nk - 1));
    int c = 0;
    for (; (c + 2) * D <= nk; ++c) chunk(c, std::true_type{});
    for (; c * D < nk; ++c) chunk(c, std::false_type{});
  }
};

// One wave streams 16 MT rows and NS weight tiles, its own part of K, through a private ring D steps deep: no barrier.
template <int MT, int NS, int D>
struct OwnRows {
  static constexpr int L = MT + NS, BYTES = D * L * 1024;

  // src: this lane's sources, weight tiles first; ns: steps
  static __device__ __forceinline__ void run(char* lds, const bf16_t* const (&src)[L], int ns, f32x4 (&acc)[MT][NS]) {
    if (ns <= 0) return;
    const int rd = piece_frag();
    auto issue = [&](int slot, int k) {
#pragma unroll
      for (int i = 0; i < L; ++i) load_piece(lds + (slot * L + i) * 1024, src[i] + 32 * k);
    };
    auto consume = [&](int slot) {
      bf16x8 f[L];
#pragma unroll
      for (int i = 0; i < L; ++i) f[i] = *reinterpret_cast<const bf16x8*>(lds + (slot * L + i) * 1024 + rd);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot may be refilled
#pragma unroll
      for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[NS + m], f[t], acc[m][t], 0, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, min(d, ns - 1));
    int slot = 0, k = 0;
    for (; k + D < ns; ++k) {
      loads_left<(D - 1) * L>();
      consume(slot);
      issue(slot, k + D);
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    auto rest = [&](auto self, auto dc) {
      constexpr int d = decltype(dc)::value;
      if constexpr (d < D) {
        loads_left<(D - 1 - d) * L>();
        if (k + d < ns) {
          consume(slot);
          slot = slot + 1 == D ? 0 : slot + 1;
        }
        self(self, std::integral_constant<int, d + 1>{});
      }
    };
    rest(rest, std::integral_constant<int, 0>{});
  }
};

}  // namespace k8sllm
