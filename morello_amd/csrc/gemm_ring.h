// What the two kernels named k_gemm_ring share: operands straight from memory into LDS (gemm_ring.hip) and through
// registers from rows that start anywhere (gemm_ring_rows.hip).
#pragma once
#include <algorithm>

#include "gemm_mfma_kernel.h"

namespace mrl {
namespace ring {
using gemm::BF16;
using gemm::I8;
using gemm::v2i;
using gemm::v4i;
using gemm::v8bf;
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int STEP = 128, WAVES = 8;   // bytes of K a step: two MFMAs deep, one for each half of the waves

template <class T> struct Ring;
template <> struct Ring<I8> {
  typedef v4i Acc;
  __device__ static Acc mfma(v4i a, v4i b, Acc c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }
};
template <> struct Ring<BF16> {
  typedef v4f Acc;
  __device__ static Acc mfma(v4i a, v4i b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
};

// Byte position of a row-major B's piece-and-rest `byte` of k row r <-> in memory (an involution).  Rows
// of BN elements; a row's place relative to the 256 bytes of a bank line repeats every 256 / (pitch % 256).
template <class T, int BN>
__device__ inline int swizzle(int byte, int r) {
  constexpr int PITCH = BN * T::ES, PIECE = 16 * T::ES;
  // the bits of the row number that tell apart the rows half a wave reads at once: bf16 r & 3 and bit 3, int8 r & 7 and bit 4
  const int rows = T::ES == 2 ? (r & 3) | ((r >> 3) & 1) << 2 : (r & 7) | ((r >> 4) & 1) << 3;
  constexpr int OFF = PITCH % 256;   // 0: all rows start in the same bank; 128 (64, 192): the low bit (two bits) of the row already moves it
  constexpr int MOVED = OFF == 0 ? 0 : OFF % 128 == 0 ? 1 : OFF % 64 == 0 ? 2 : 3;
  constexpr int PIECES = (256 >> MOVED) / PIECE;   // of a group to exchange within
  const int x = (rows >> MOVED) & (PIECES - 1);
  return ((byte / PIECE) ^ x) * PIECE + byte % PIECE;
}

constexpr int divisor_up_to(int most, int n) { return n % most == 0 ? most : divisor_up_to(most - 1, n); }
constexpr int min_of(int a, int b) { return a < b ? a : b; }
// f(0), ..., f(N - 1) with the number as a type
template <int N, int I = 0, class F>
__device__ __forceinline__ void each(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<N, I + 1>(f);
  }
}

// C from the sums of a tile's eight waves: RA x RB blocks of 16 x 16 each, the waves wm, wn of the first (kw = 0) and
// second half of every step.  `skip`: columns of the tile, from its first, that are another tile's.
template <class T, bool A_UNSIGNED, int RA, int RB>
__device__ __forceinline__ void store_tile(const GemmArgs &g, uint8_t *lds, typename Ring<T>::Acc (&acc)[RA][RB], int (&colsum)[RB],
                                           int64_t m0, int64_t n0, int skip) {
  typedef typename T::Out Out;
  constexpr int WM = 16 * RA, WN = 16 * RB;
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kw = wave >> 2, wm = wave >> 1 & 1, wn = wave & 1;
  // C.  Register i of a block: row 4 (l / 16) + i, column l % 16.  A wave's block row goes through its own
  // piece of LDS and leaves in whole rows of WN columns.
  if (A_UNSIGNED)
#pragma unroll
    for (int c = 0; c < RB; c++) {
      colsum[c] += __shfl_xor(colsum[c], 16);
      colsum[c] += __shfl_xor(colsum[c], 32);
      colsum[c] *= 128;
    }
  constexpr int ROW = WN + 4;
  Out *piece = (Out *)lds + (wave & 3) * (WM * ROW);
  const int64_t row_first = m0 + wm * WM, col_first = n0 + wn * WN;
  const int cols = int(min(int64_t(WN), int64_t(g.n) - col_first));
  const int from = skip - wn * WN;   // of this wave's columns
  // (The loops stay loops: code that a launch runs once is fetched from memory, and unrolled it took longer to
  // fetch than to run.)
  auto store = [&](auto *C) {
    typedef std::remove_pointer_t<decltype(C)> Stored;
    C += int64_t(blockIdx.y) * g.sc + row_first * g.ldc + col_first;
    const int rows = int(min(int64_t(WM), int64_t(g.m) - row_first));
    const int some = max(from, 0);   // a place of this wave's: read, not written, by lanes that have none
    // An element a lane, or four where all of a row's columns are whole and aligned.  Of bf16 eight where they are not, wherever rows start: two bytes a
    // lane take as many accesses to an eighth of the bytes (us, by elements / eights: 1501 x 1001 x 2001 18.5 / 17.2, 2072 x 1899 x 2689 36.4 / 33.9, 179 x 142
    // x 2617 4.3 / 4.0, 1001 x 2050 x 4425 with its copies 35.8 / 33.9; onto old values, eights read from anywhere too, 1500 x 300 x 1501 11.0 / 14.6).
    // Old values come in batches: one at a time, each behind the store before it, they took longer than a short K (bf16 2163 x 420 x 513).
    auto rows_of = [&](auto at_once) {
      constexpr int V = decltype(at_once)::value, COUNT = (WM * WN / V + 127) / 128, BATCH = divisor_up_to(8, COUNT);
      typedef Stored stored_v __attribute__((ext_vector_type(V)));
      typedef stored_v stored_there __attribute__((aligned(V == 8 ? sizeof(Stored) : V * sizeof(Stored))));
      typedef Out out_v __attribute__((ext_vector_type(V)));
      typedef out_v out_there __attribute__((aligned(V < 4 ? 4 : 16)));
#pragma unroll 1
      for (int e = 0; e < COUNT; e += BATCH) {
        int64_t to[BATCH];
        out_v v[BATCH];
        stored_v old[BATCH];
        bool mine[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
          const int at = (2 * (e + u) + kw) * 64 + lane, row = at / (WN / V), col = at % (WN / V) * V;
          mine[u] = row < rows && col >= from && (V == 8 ? col + V <= cols : col < cols);
          to[u] = mine[u] ? int64_t(row) * g.ldc + col : some;
          v[u] = *(const out_there *)(piece + (V == 8 ? min(row, WM - 1) : row) * ROW + col);
          if constexpr (V == 8)
            if (!mine[u] && row < rows)   // what an edge cuts
#pragma unroll 1
              for (int c = max(col, from); c < min(col + V, cols); c++) C[int64_t(row) * g.ldc + c] = Stored(piece[row * ROW + c]);
        }
        if (V < 8 && g.accum) {
#pragma unroll
          for (int u = 0; u < BATCH; u++) old[u] = *(const stored_there *)(C + to[u]);
#pragma unroll
          for (int u = 0; u < BATCH; u++) v[u] += __builtin_convertvector(old[u], out_v);
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++)
          if (mine[u]) *(stored_there *)(C + to[u]) = __builtin_convertvector(v[u], stored_v);
      }
    };
    if (cols % 4 == 0 && from % 4 == 0 && g.ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C) % (4 * sizeof(Stored)) == 0) rows_of(std::integral_constant<int, 4>{});
    else if (sizeof(Stored) == 2 && !g.accum) rows_of(std::integral_constant<int, sizeof(Stored) == 2 ? 8 : 1>{});
    else rows_of(std::integral_constant<int, 1>{});
  };
  // The two halves of K: the upper waves' sums through LDS onto the lower waves', and both store.
  auto for_each_sum = [&](auto f) {
#pragma unroll
    for (int r = 0; r < RA; r++)
#pragma unroll
      for (int c = 0; c < RB; c++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          Out v = acc[r][c][i];
          if (A_UNSIGNED) v += Out(colsum[c]);
          f(piece[(r * 16 + 4 * lg + i) * ROW + c * 16 + li], v);
        }
  };
  if (kw) for_each_sum([](Out &at, Out v) { at = v; });
  __syncthreads();
  if (!kw) for_each_sum([](Out &at, Out v) { at = v + at; });
  __syncthreads();
  if (cols > max(from, 0) && row_first < int64_t(g.m)) {
    if constexpr (std::is_same<T, BF16>::value) {
      if (g.c_bf16) store((__bf16 *)g.c);
      else store((Out *)g.c);
    } else store((Out *)g.c);
  }
}

}  // namespace ring
}  // namespace mrl
