// The tile of gemm_ring_rows.hip: rows that start anywhere.
#pragma once
#include "gemm_ring.h"

namespace mrl {
namespace ring {
typedef int chunk_anywhere __attribute__((ext_vector_type(4), aligned(1)));
typedef __attribute__((address_space(1))) const uint8_t global_u8;
typedef __attribute__((address_space(1))) const chunk_anywhere global_chunk;

// The first `left` of v's bytes (none below 1, all from 16 on), zeros behind them.
__device__ inline v4i first_bytes(v4i v, int left) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int n = left - 4 * i;
    v[i] &= n >= 4 ? -1 : n <= 0 ? 0 : int((1u << (8 * n)) - 1);
  }
  return v;
}

template <class T, bool A_UNSIGNED, bool B_KMAJOR, int RA, int RB>
__device__ __forceinline__ void rows_tile(uint8_t *lds, uint32_t tile_m, uint32_t tile_n, const GemmArgs &g) {
  typedef typename Ring<T>::Acc Acc;
  constexpr int ES = T::ES, BK = STEP / ES, BM = 32 * RA, BN = 32 * RB, WM = 16 * RA, WN = 16 * RB;
  constexpr int A_BYTES = BM * STEP, B_BYTES = BN * STEP, SLOT = A_BYTES + B_BYTES;
  constexpr int A_LOADS = A_BYTES / (1024 * WAVES), B_LOADS = (B_BYTES / 1024 + WAVES - 1) / WAVES, LOADS = A_LOADS + B_LOADS;   // a wave's, per step
  // The k loop in pairs of steps and one more.  With an exit between the two, the other form, the compiler sees a way from the first to itself and makes
  // it wait for all but half a step's loads: less code, and as good as or better than two whole steps under way on 128 x 128 tiles and, of int8 along K,
  // wider ones (u8 726 x 996 x 4035 12.9 / 13.4, 2432 x 1702 x 2069 25.2 / 25.6).  Else worse: bf16 138 x 699 x 368 6.6 / 6.2, 394 x 139 x 145 5.0 / 4.5.
  constexpr bool PAIRS = RB < 4 || (RB > 4 && !(ES == 1 && B_KMAJOR));
  // Steps of loads under way (four to eight, on the smallest tile: 4 to 13 % slower, more to wait for at the start and nothing gained behind it).  In
  // pairs on the widest tiles rows of any alignment lose by the second (bf16 2306 x 735 x 2260 17.3 us, with one 17.0; 3456 x 1909 x 1221 32.9 / 32.4).
  constexpr int DEPTH = PAIRS && RB >= 5 ? 1 : 2;
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kw = wave >> 2, wm = wave >> 1 & 1, wn = wave & 1;
  const int64_t m0 = int64_t(tile_m) * BM, n_tile = int64_t(tile_n) * BN;
  const int64_t n0 = B_KMAJOR ? n_tile : min(n_tile, int64_t(g.n) - BN);
  const uint8_t *A = (const uint8_t *)g.a + (int64_t(blockIdx.y) * g.sa + m0 * g.lda) * ES;
  const uint8_t *B = (const uint8_t *)g.b + (int64_t(blockIdx.y) * g.sb + (B_KMAJOR ? n0 * g.ldb : n0)) * ES;
  const uint32_t lda_b = uint32_t(g.lda) * ES, ldb_b = uint32_t(g.ldb) * ES;
  const int a_last = min(BM, int(g.m - m0)) - 1, b_last = min(BN, int(g.n - n0)) - 1;
  const int k = g.k_total != 0 ? int(min(g.k, g.k_total - blockIdx.y * g.k)) : int(g.k), steps = (k + BK - 1) / BK, head = k - (steps - 1) * BK;   // head: elements of K in the first step

  // Where this lane's chunks of a step come from, as in gemm_ring.hip: lane l of a load has the l-th 16 bytes of a KiB of LDS.
  auto b_load = [&](int i) { return i * WAVES + wave - (i * WAVES + wave < B_BYTES / 1024 ? 0 : WAVES / 2); };
  constexpr int CHUNKS = STEP / 16, ROWS_PER_LOAD = 64 / CHUNKS, ROWS_PER_LINE = 256 / STEP;
  const int row16 = lane / CHUNKS, chunk = (lane % CHUNKS) ^ (row16 / ROWS_PER_LINE % CHUNKS);
  auto chunk_of = [&](int load) { return chunk ^ (load * ROWS_PER_LOAD / ROWS_PER_LINE % CHUNKS); };
  uint32_t off[LOADS];
  int dst[LOADS], whole[LOADS];   // whole: of the chunk's 16 bytes, those the first step has
#pragma unroll
  for (int i = 0; i < A_LOADS; i++) {
    const int load = wave * A_LOADS + i;
    off[i] = uint32_t(min(load * ROWS_PER_LOAD + row16, a_last)) * lda_b + chunk_of(load) * 16;
    dst[i] = load * 1024 + lane * 16;
    whole[i] = head * ES - chunk_of(load) * 16;
  }
#pragma unroll
  for (int i = 0; i < B_LOADS; i++) {
    const int load = b_load(i);
    dst[A_LOADS + i] = A_BYTES + load * 1024 + lane * 16;
    if constexpr (B_KMAJOR) {
      off[A_LOADS + i] = uint32_t(min(load * ROWS_PER_LOAD + row16, b_last)) * ldb_b + chunk_of(load) * 16;
      whole[A_LOADS + i] = head * ES - chunk_of(load) * 16;
    } else {
      constexpr int PITCH = BN * ES;
      const int at = load * 1024 + lane * 16, r = at / PITCH;
      off[A_LOADS + i] = uint32_t(r) * ldb_b + swizzle<T, BN>(at % PITCH, r);
      whole[A_LOADS + i] = r < head ? 16 : 0;
    }
  }
  const global_u8 *a_tile = (const global_u8 *)A, *b_tile = (const global_u8 *)B;
  const int64_t b_step = B_KMAJOR ? int64_t(STEP) : int64_t(BK) * ldb_b;
  auto load = [&](auto which) {
    constexpr int I = decltype(which)::value;
    return __builtin_bit_cast(v4i, *(const global_chunk *)((I < A_LOADS ? a_tile : b_tile) + off[I]));
  };
  int behind = steps;   // steps from the one that the pointers are at on
  // To the next one (past the last: nowhere); `first`: from the first step, which has `head` elements.
  auto advance = [&](auto first) {
    const bool more = --behind > 0;
    const int a_step = !more ? 0 : decltype(first)::value ? head * ES : STEP;
    a_tile += a_step;
    if constexpr (PAIRS) asm("" : "+s"(a_tile));   // (scalar bases, not sums of each lane's)
    b_tile += !more ? 0 : !decltype(first)::value ? b_step : B_KMAJOR ? int64_t(head) * ES : int64_t(head) * ldb_b;
    if constexpr (PAIRS) asm("" : "+s"(b_tile));
  };

  // Operand addresses within a slot: lane (l % 16, l / 16) takes the l / 16-th 16 bytes of row l % 16.
  const int in_rows = li * STEP + (((4 * kw + lg) ^ (li / ROWS_PER_LINE % CHUNKS)) << 4);
  int b_rd[RB];
  if constexpr (!B_KMAJOR) {
    constexpr int LANES_PER_ROW = 2 * ES;   // of a group of sixteen: 8 bytes each of a row's sixteen columns
    const int r = (64 / ES) * kw + (16 / ES) * lg + li / LANES_PER_ROW;
#pragma unroll
    for (int c = 0; c < RB; c++) b_rd[c] = A_BYTES + r * (BN * ES) + swizzle<T, BN>((wn * WN + c * 16) * ES + 8 * (li % LANES_PER_ROW), r);
  }
  v4i af[2][RA], bf[2][RB], kept[DEPTH][LOADS];
  // The i-th operand read of 64 bytes of K (RA of A, then RB of B), out of the slot of the same parity.
  auto read = [&](auto set, auto which) {
    constexpr int S = decltype(set)::value, I = decltype(which)::value;
    const uint8_t *slot = lds + S * SLOT;
    if constexpr (I < RA) af[S][I] = *(const v4i *)(slot + wm * WM * STEP + in_rows + I * 16 * STEP);
    else if constexpr (B_KMAJOR) bf[S][I - RA] = *(const v4i *)(slot + A_BYTES + wn * WN * STEP + in_rows + (I - RA) * 16 * STEP);
    else {
      const uint8_t *at = slot + b_rd[I - RA];
      const v2i lo = T::read_tr(at), hi = T::read_tr(at + T::K_PER_READ * (BN * ES));
      bf[S][I - RA] = v4i{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  Acc acc[RA][RB];
  int colsum[RB];
#pragma unroll
  for (int c = 0; c < RB; c++) {
    colsum[c] = 0;
#pragma unroll
    for (int r = 0; r < RA; r++) acc[r][c] = Acc{0, 0, 0, 0};
  }
  auto multiply = [&](auto set, auto which) {   // the which-th block
    constexpr int S = decltype(set)::value, I = decltype(which)::value, R = I / RB, C = I % RB;
    if constexpr (A_UNSIGNED && C == 0) af[S][R] ^= v4i{int(0x80808080), int(0x80808080), int(0x80808080), int(0x80808080)};
    acc[R][C] = Ring<T>::mfma(af[S][R], bf[S][C], acc[R][C]);
    if constexpr (A_UNSIGNED && R == 0)   // a - 128 was multiplied: 128 times the column sums of B come on top
#pragma unroll
      for (int w = 0; w < 4; w++) colsum[C] = __builtin_amdgcn_sdot4(bf[S][C][w], 0x01010101, colsum[C], false);
  };
  // All LDS reads and writes are done; loads stay under way.  (A builtin wait, which the compiler sees: it adds none of its own for the operands that are in.)
  auto barrier = [] {
    asm volatile("" : : : "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
  };
  // A step of parity P whose successor but one waits in set K.
  auto step = [&](auto parity, auto held) {
    constexpr int P = decltype(parity)::value, K = decltype(held)::value;
    barrier();
    each<RA * RB>([&](auto q) {
      constexpr int Q = decltype(q)::value, N = RA * RB, READS = RA + RB;
      multiply(parity, q);
      constexpr int R0 = min_of(READS, (Q * READS * 4 + N * 3 - 1) / (N * 3)), R1 = min_of(READS, ((Q + 1) * READS * 4 + N * 3 - 1) / (N * 3));   // in the first three quarters
      each<R1 - R0>([&](auto i) { read(std::integral_constant<int, 1 - P>{}, std::integral_constant<int, R0 + decltype(i)::value>{}); });
      constexpr int L0 = Q * LOADS / N, L1 = (Q + 1) * LOADS / N;
      each<L1 - L0>([&](auto i) {
        constexpr int I = L0 + decltype(i)::value;
        *(v4i *)(lds + P * SLOT + dst[I]) = kept[K][I];
        kept[K][I] = load(std::integral_constant<int, I>{});
      });
      if constexpr (Q == N - 1) advance(std::false_type{});
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  {
    v4i first[2][LOADS];
    each<2>([&](auto s) {
      each<LOADS>([&](auto i) { first[decltype(s)::value][decltype(i)::value] = load(i); });
      if constexpr (PAIRS) __builtin_amdgcn_sched_barrier(0);
      advance(std::integral_constant<bool, decltype(s)::value == 0>{});
    });
    each<DEPTH>([&](auto s) {
      each<LOADS>([&](auto i) {
        kept[decltype(s)::value][decltype(i)::value] = load(i);
        if constexpr (PAIRS) __builtin_amdgcn_sched_barrier(0);   // in this order, which the loop's waits count on
      });
      advance(std::false_type{});
    });
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
      *(v4i *)(lds + dst[i]) = first_bytes(first[0][i], whole[i]);
      *(v4i *)(lds + SLOT + dst[i]) = first[1][i];
    }
  }
  barrier();
  each<RA + RB>([&](auto i) { read(std::integral_constant<int, 0>{}, i); });
  // (What a step reads and writes for those behind the last one is not multiplied.)
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  const std::integral_constant<int, DEPTH - 1> second;
  if constexpr (!PAIRS) {
    for (int left = steps;;) {
      bool done = false;
      each<2>([&](auto s) {
        if (!done) {
          step(s, std::integral_constant<int, decltype(s)::value % DEPTH>{});
          done = --left == 0;
        }
      });
      if (done) break;
    }
  } else {
    for (int left = steps; left >= 2; left -= 2) {
      step(even, even);
      step(odd, second);
    }
    if (steps & 1) step(even, even);
  }
  barrier();
  store_tile<T, A_UNSIGNED, RA, RB>(g, lds, acc, colsum, m0, n0, int(n_tile - n0));
}

}  // namespace ring
}  // namespace mrl
