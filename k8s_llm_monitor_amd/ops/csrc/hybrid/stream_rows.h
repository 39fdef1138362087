// Weight streams for a few rows: 16 output columns a wave, everything that v_mfma_f32_16x16x32_bf16 takes brought to LDS by
// global_load_lds, 16 bytes a lane, in lines of 16 rows x 64 k (windowed attention's keys in pieces of 16 rows x 32 k).
// Why LDS and not registers: the instruction wants row lane % 16 in a lane, so a register load of row-major rows meets 16 cache lines in
// every 16 lanes and takes about 60 cycles of the load path (512 KB from L2 by one CU: 13 us, 3.6 us in lane order), and activations take as
// much of it as weights do.
// A piece (1 KB) has four lanes a row; the chunk that lane l fetches is turned by the row, so that the
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
// the same for what a step reads once: non-temporal, so that it does not push out what is read again
__device__ __forceinline__ void load_piece_once(char* lds, const bf16_t* src) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) const void*)src, (__attribute__((address_space(3))) void*)lds, 16,
                                   0, 2);
}
template <int N>
__device__ __forceinline__ void loads_left() {  // waits until at most N of this wave's loads are on their way
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// A line: 16 rows x 64 k, 2 KB, two loads of 8 rows in whole 128-byte cache lines (a piece's 64 bytes a row ask for every cache line
// twice).  us over weights from memory, in pieces / in lines / in lines with the weights non-temporal, few_rows.hip: 4096 x 4096, 64 rows
// 19.9 / 14.1 / 13.6; 16384 x 4096, 1 row 26.3 / 26.9 / 23.6, 64 rows 36.3 / 34.7 / 30.8; 128256 x 4096, 1 row 179 / 186 / 162 (6.5 TB/s);
// 1024 x 1024, 1 row 2.9 / 3.0 / 3.1; 8 experts of 2048 x 2048, gated, 128 rows 36.9 / 35.1 / 31.9, 800 rows 47.7 / 42.9 / 41.7.  Twice the
// lines in flight gain nothing anywhere.
// The weights of a call of up to 8 MB are loaded as usual (kOnceBytes): a model of such calls has its place in the memory-side cache of 256 MB.
// Steps of one sequence with 2 of 8 experts of 1024 x 1024 in four layers, us: never / always / above 8 MB non-temporal 245 / 250 / 244, of 64 424 /
// 383 / 380.
// Load i of lane l brings row 8 i + l / 8, and of its eight 16-byte chunks the one that is turned by row / 2: sixteen
// rows' fragments of one k are then sixteen different chunks of 256 bytes.
__device__ __forceinline__ int line_row(int i) { return 8 * i + ((threadIdx.x & 63) >> 3); }
__device__ __forceinline__ int line_k(int i) { return 8 * ((threadIdx.x & 7) ^ (4 * i + ((threadIdx.x & 63) >> 4))); }
__device__ __forceinline__ int line_frag() {  // of a line's first 32 k; the others' are at ^ 64
  const int lane = threadIdx.x & 63, c16 = lane & 15;
  return c16 * 128 + 16 * ((lane >> 4) ^ (c16 >> 1));
}
// Where this lane finds its chunks of a line's two loads, at k = 0.  K ends inside a line if it is an odd number of 32: the chunks behind
// it, and lines behind the last, are read from the row's last chunk, and nothing multiplies them.
// Rows that do not begin at a cache line (an odd number of 32 k) too: two loads meet each of their lines, and what the first brought has gone
// before the second (4704 k, 1968 columns, 3 rows 7.5 / 7.15, 15 of them in turn 8.8 / 6.6; 928 k, 19776 columns, 1 row 9.9 / 9.7, 11.4 / 10.5; 4128 k,
// 4096 columns, 1 row 8.1 / 8.3, 9.9 / 9.3).
constexpr long kOnceBytes = 8l << 20;
inline bool read_once(long bytes, const void* w, int kd) {
  return bytes > kOnceBytes && kd % 64 == 0 && reinterpret_cast<uintptr_t>(w) % 128 == 0;
}
struct LineSrc {
  const bf16_t* p[2];
  __device__ __forceinline__ int within(int i, int k, int kd) const { return min(k, kd - 8 - line_k(i)); }
  __device__ __forceinline__ void load(char* lds, int i, int k) const { load_piece(lds + 1024 * i, p[i] + k); }
  __device__ __forceinline__ void once(char* lds, int i, int k) const { load_piece_once(lds + 1024 * i, p[i] + k); }
};
// Where workgroup b begins among n pieces of its rows, so that those that run side by side are not at the same k: with rows of weights whole
// periods of the channels apart (4 KB), every workgroup's lines of one k lie in the same channels of its XCD's L2 and of memory.  us, all from k = 0 /
// so: shared form, 24 rows 16384 x 4096 28.8 / 24.9, 65536 x 4096 99 / 87, 16 rows 16384 x 6144 43 / 36, 65536 x 10240 227 / 209; of rows of one period
// 8192 x 2048 11.9 / 11.5, 32000 x 2048 27.4 / 26.5, 64 rows 34.3 / 32.2, 24 rows 10240 x 2048 12.2 / 12.2; own form, 1 row 4096 x 16384 28.3 / 23.8, 4096 x 8192
// 15.6 / 14.5, 8192 x 8192 27.2 / 26.0; 16384 x 4160, which needs it not, 23.3.  Few workgroups do not meet and lose a little: 1 row 1024 x 16384 14.9 / 15.5,
// 512 x 16384 14.0 / 14.3.  The order of the fp32 sums follows it: what must keep its sums' order begins at 0.
constexpr int kTurnBytes = 4096, kTurnGroups = 128;
__device__ __forceinline__ int first_piece(int b, int n) { return ((b >> 3) + (b & 7)) % n; }
// row(r): where row r (of 16) begins
template <class R>
__device__ __forceinline__ LineSrc line_src(R row) {
  return {{row(line_row(0)) + line_k(0), row(line_row(1)) + line_k(1)}};
}

// NW waves of one workgroup share 16 MT rows, which come in chunks of 4 lines to a ring of two; each wave streams its own NS
// weight tiles through a private ring, 4 lines ahead.  Every output is one chain of products in the order of k.  ONCE: the
// weights' loads are non-temporal.
template <int MT, int NS, int NW, bool ONCE, bool TURN = false>
struct SharedRows {
  static constexpr int D = 4;  // lines of a chunk, and of the weights' ring
  static constexpr int SLOT = D * MT * 2048, RING = D * NS * 2048, BYTES = 2 * SLOT + NW * RING;
  // a wave brings one row tile's loads of a chunk: all, those of every line's half, or those of every other line's half
  static constexpr int P = NW / MT, PER = 2 * D / P, HALVES = P == 1 ? 2 : 1, EVERY = P > 2 ? P / 2 : 1;
  static_assert(NW % MT == 0 && P <= 4, "");

  // x(m): this lane's sources in row tile m of the rows; w[t]: in weight tile t; kd: a multiple of 32; TURN: of whole
  // chunks, of which c0 is the first to be taken (first_piece)
  template <class X>
  static __device__ __forceinline__ void run(char* lds, X x, const LineSrc (&w)[NS], int kd, f32x4 (&acc)[MT][NS], int c0 = 0) {
    const int nc = kd / (64 * D);
    auto at = [&](int c) { return !TURN ? c : c + c0 >= nc ? c + c0 - nc : c + c0; };
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rd = line_frag(), nl = (kd + 63) / 64;
    const int m0 = wave % MT, h0 = (wave / MT) & (P > 1 ? 1 : 0), u0 = P > 2 ? wave / MT / 2 : 0;
    const LineSrc xs = x(m0);
    char* ring = lds + 2 * SLOT + wave * RING;
    auto stage = [&](int c, auto whole) {
#pragma unroll
      for (int i = 0; i < D / EVERY; ++i)
#pragma unroll
        for (int j = 0; j < HALVES; ++j) {
          const int u = u0 + i * EVERY, h = HALVES == 1 ? h0 : j;
          const int k = 64 * (at(c) * D + u);
          load_piece(lds + (c & 1) * SLOT + (u * MT + m0) * 2048 + 1024 * h,
                     (h ? xs.p[1] : xs.p[0]) + (decltype(whole)::value ? k : xs.within(h, k, kd)));
        }
    };
    auto refill = [&](int u, int c, auto whole) {
      const int l = at(c) * D + u;
#pragma unroll
      for (int t = 0; t < NS; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int k = decltype(whole)::value ? 64 * l : w[t].within(i, 64 * l, kd);
          if constexpr (ONCE) w[t].once(ring + (u * NS + t) * 2048, i, k);
          else w[t].load(ring + (u * NS + t) * 2048, i, k);
        }
    };
    auto chunk = [&](int c, auto whole) {
      constexpr bool WHOLE = decltype(whole)::value;  // every line, the next chunk and every refill are inside K
      if constexpr (WHOLE) loads_left<2 * D * NS>();  // the chunk's loads are older than the ring's
      else loads_left<0>();
      __builtin_amdgcn_s_barrier();  // every wave's loads are there, and the other slot has been read
      if (WHOLE || (c + 1) * D < nl) stage(c + 1, whole);
      auto line = [&](auto self, auto uc) {
        constexpr int u = decltype(uc)::value;
        if constexpr (u < D) {
          if (WHOLE || c * D + u < nl) {
            // younger than this line's weights: the D - 1 lines behind it and the chunk just begun
            if constexpr (WHOLE) loads_left<2 * (D - 1) * NS + PER>();
            else if (u > 0) loads_left<0>();
            bf16x8 a[2][MT], b[2][NS];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
              for (int t = 0; t < NS; ++t) b[j][t] = *reinterpret_cast<const bf16x8*>(ring + (u * NS + t) * 2048 + (rd ^ (64 * j)));
#pragma unroll
              for (int m = 0; m < MT; ++m)
                a[j][m] = *reinterpret_cast<const bf16x8*>(lds + (c & 1) * SLOT + (u * MT + m) * 2048 + (rd ^ (64 * j)));
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (WHOLE || (c + 1) * D + u < nl) refill(u, c + 1, whole);
#pragma unroll
            for (int j = 0; j < 2; ++j)
              if (j == 0 || WHOLE || 64 * (c * D + u) + 32 < kd) {
#pragma unroll
                for (int t = 0; t < NS; ++t)
#pragma unroll
                  for (int m = 0; m < MT; ++m) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][m], b[j][t], acc[m][t], 0, 0, 0);
              }
          }
          __builtin_amdgcn_sched_barrier(0);
          self(self, std::integral_constant<int, u + 1>{});
        }
      };
      line(line, std::integral_constant<int, 0>{});
    };
    stage(0, std::false_type{});
#pragma unroll
    for (int u = 0; u < D; ++u) refill(u, 0, std::false_type{});
    int c = 0;
    for (; 64 * (c + 2) * D <= kd; ++c) chunk(c, std::true_type{});
    for (; c * D < nl; ++c) chunk(c, std::false_type{});
  }
};

// One wave streams 16 MT rows and NS weight tiles, its own part of K, through a private ring D lines deep: no barrier.
template <int MT, int NS, int D, bool ONCE, bool TURN = false>
struct OwnRows {
  static constexpr int L = MT + NS, BYTES = D * L * 2048;

  // src: this lane's sources, weight tiles first; kd: k of this part, a multiple of 32; TURN: of whole lines, of
  // which l0 is the first to be taken (first_piece)
  static __device__ __forceinline__ void run(char* lds, const LineSrc (&src)[L], int kd, f32x4 (&acc)[MT][NS], int l0 = 0) {
    if (kd <= 0) return;
    const int rd = line_frag(), nl = (kd + 63) / 64;
    auto at = [&](int l) { return !TURN || l >= nl ? l : l + l0 >= nl ? l + l0 - nl : l + l0; };
    auto issue = [&](int slot, int line, auto whole) {
      const int l = at(line);
#pragma unroll
      for (int i = 0; i < L; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int k = decltype(whole)::value ? 64 * l : src[i].within(j, 64 * l, kd);
          if (ONCE && i < NS) src[i].once(lds + (slot * L + i) * 2048, j, k);
          else src[i].load(lds + (slot * L + i) * 2048, j, k);
        }
    };
    auto consume = [&](int slot, bool half) {
      bf16x8 f[2][L];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < L; ++i) f[j][i] = *reinterpret_cast<const bf16x8*>(lds + (slot * L + i) * 2048 + (rd ^ (64 * j)));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot may be refilled
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (j == 0 || !half) {
#pragma unroll
          for (int t = 0; t < NS; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[j][NS + m], f[j][t], acc[m][t], 0, 0, 0);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, d, std::false_type{});
    int slot = 0, l = 0;
    for (; 64 * (l + D + 1) <= kd; ++l) {
      loads_left<2 * (D - 1) * L>();
      consume(slot, false);
      issue(slot, l + D, std::true_type{});
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    if (l + D < nl) {  // the line that K ends in
      loads_left<2 * (D - 1) * L>();
      consume(slot, false);
      issue(slot, l + D, std::false_type{});
      slot = slot + 1 == D ? 0 : slot + 1;
      ++l;
    }
    auto rest = [&](auto self, auto dc) {
      constexpr int d = decltype(dc)::value;
      if constexpr (d < D) {
        loads_left<2 * (D - 1 - d) * L>();
        if (l + d < nl) {
          consume(slot, 64 * (l + d) + 32 >= kd);
          slot = slot + 1 == D ? 0 : slot + 1;
        }
        self(self, std::integral_constant<int, d + 1>{});
      }
    };
    rest(rest, std::integral_constant<int, 0>{});
  }
};

// The same with rows that lie in LDS whole (up to 16 of them, row r's k at xs + r * pitch; rows past the last read the last): only weights are
// streamed.  begin() sends the first D lines on their way, run() takes them all.
template <int NS, int D, bool ONCE>
struct HeldRows {
  static constexpr int BYTES = D * NS * 2048;

  static __device__ __forceinline__ void issue(char* lds, const LineSrc (&w)[NS], int slot, int l, int kd) {
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int k = w[t].within(j, 64 * l, kd);
        if constexpr (ONCE) w[t].once(lds + (slot * NS + t) * 2048, j, k);
        else w[t].load(lds + (slot * NS + t) * 2048, j, k);
      }
  }
  static __device__ __forceinline__ void begin(char* lds, const LineSrc (&w)[NS], int kd) {
    if (kd <= 0) return;
#pragma unroll
    for (int d = 0; d < D; ++d) issue(lds, w, d, d, kd);
  }
  // x: this lane's row, at the first k of its chunk (lane / 16) of this part
  static __device__ __forceinline__ void run(char* lds, const LineSrc (&w)[NS], const bf16_t* x, int kd, f32x4 (&acc)[NS]) {
    if (kd <= 0) return;
    const int rd = line_frag(), nl = (kd + 63) / 64;
    int slot = 0;
    auto consume = [&](int l) {
      bf16x8 b[2][NS], a[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        a[j] = *reinterpret_cast<const bf16x8*>(x + min(64 * l + 32 * j, kd - 32));
#pragma unroll
        for (int t = 0; t < NS; ++t) b[j][t] = *reinterpret_cast<const bf16x8*>(lds + (slot * NS + t) * 2048 + (rd ^ (64 * j)));
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot may be refilled
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (j == 0 || 64 * l + 32 < kd) {
#pragma unroll
          for (int t = 0; t < NS; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j], b[j][t], acc[t], 0, 0, 0);
        }
    };
    int l = 0;
    for (; l + D < nl; ++l) {
      loads_left<2 * (D - 1) * NS>();
      consume(l);
      issue(lds, w, slot, l + D, kd);
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    auto rest = [&](auto self, auto dc) {
      constexpr int d = decltype(dc)::value;
      if constexpr (d < D) {
        loads_left<2 * (D - 1 - d) * NS>();
        if (l + d < nl) {
          consume(l + d);
          slot = slot + 1 == D ? 0 : slot + 1;
        }
        self(self, std::integral_constant<int, d + 1>{});
      }
    };
    rest(rest, std::integral_constant<int, 0>{});
  }
};

}  // namespace k8sllm
