// The tile of gemm_ring.hip: rows of whole 16-byte chunks, or (CONV) the windows of a channels-last image of such pixels.
#pragma once
#include "gemm_ring.h"
#include "tile_bounds.h"

namespace mrl {
namespace ring {
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) const uint8_t lds_u8;
typedef __attribute__((address_space(3))) const v4i lds_v4i;

constexpr uint32_t OUTSIDE = 0xf0000000u;   // an offset no resource here holds: 192 rows of 2^24 bytes, an image of 2^31

// One load of 64 lanes x 16 bytes into the KiB at LDS address `lds_addr` + AT (wave-uniform), lane l to the l-th
// 16 bytes; the instruction's offset AT is added to the address in memory too, so callers take it off
// there.  An offset outside the resource brings zeros.  Assembly, so that the compiler does not wait for it; M0 is set in
// the same statement, with the wait state it needs: the compiler sets that reserved register right before its own
// uses and keeps nothing in it, and may do so between any two statements.
template <int AT>
__device__ inline void dma16(v4i from, uint32_t off, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen offset:%3 lds" : : "v"(off), "s"(from), "s"(lds_addr), "n"(AT) : "memory");
}
// (of addresses below 2^48, as all are: the bits above belong to the stride)
__device__ inline v4i resource(uint64_t base, uint32_t bytes) { return v4i{int(uint32_t(base)), int(uint32_t(base >> 32)), int(bytes), 0x00020000}; }
// All but the newest N loads have landed, and every LDS read is done.
// (A builtin wait, which the compiler sees: it adds none of its own for the operands that are in.)
template <int N>
__device__ inline void wait_for_all_but() {
  asm volatile("" : : : "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4) << 14 | 7 << 4);
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}

// CONV (with B_KMAJOR): row p of A is the window of output pixel p, fh runs of fw * c contiguous elements of the image, whole 16-byte chunks each.
template <class T, bool A_UNSIGNED, bool B_KMAJOR, int RA, int RB, int SLOTS, bool CONV = false>
__device__ __forceinline__ void ring_tile(uint8_t *lds, uint32_t tile_m, uint32_t tile_n, const GemmArgs &g) {
  static_assert(!CONV || B_KMAJOR, "");
  typedef typename Ring<T>::Acc Acc;
  constexpr int ES = T::ES, BK = STEP / ES, BM = 32 * RA, BN = 32 * RB, WM = 16 * RA, WN = 16 * RB;
  constexpr int A_BYTES = BM * STEP, B_BYTES = BN * STEP, SLOT = A_BYTES + B_BYTES;
  constexpr int A_LOADS = A_BYTES / (1024 * WAVES), B_LOADS = (B_BYTES / 1024 + WAVES - 1) / WAVES, LOADS = A_LOADS + B_LOADS;   // a wave's, per step
  static_assert((SLOTS - 1) * LOADS < 64 && A_LOADS <= 4 && B_LOADS <= 4, "");
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kw = wave >> 2, wm = wave >> 1 & 1, wn = wave & 1;
  const int64_t m0 = int64_t(tile_m) * BM, n0 = int64_t(tile_n) * BN;
  const uint8_t *A = (const uint8_t *)g.a + (CONV ? 0 : (int64_t(blockIdx.y) * g.sa + m0 * g.lda) * ES);
  const bool panels = !B_KMAJOR && g.b_panel_rows != 0;
  const uint8_t *B = (const uint8_t *)g.b + (int64_t(blockIdx.y) * g.sb + (B_KMAJOR ? n0 * g.ldb : panels ? n0 * g.b_panel_rows : n0)) * ES;
  const uint32_t lda_b = uint32_t(g.lda) * ES, ldb_b = panels ? BN * ES : uint32_t(g.ldb) * ES;
  // Bytes of the tile's rows (leading dimensions stay below 2^24 bytes); of `rows` rows of a row-major B (tile_bounds.h).
  const int a_end = min(BM, int(g.m - m0)) * int(lda_b), n_left = min(BN, int(g.n - n0));
  const uint32_t b_end = uint32_t(n_left) * ldb_b;
  auto b_rows = [&](int rows) { return uint32_t(tile_bytes(rows, ldb_b, n_left * ES)); };
  const int k = g.k_total != 0 ? int(min(g.k, g.k_total - blockIdx.y * g.k)) : int(g.k), k_bytes = k * ES, steps = (k_bytes + STEP - 1) / STEP;

  // Where this lane's chunks of a step come from.  Rows of 64 bytes: sixteen to a load.
  uint32_t a_off[A_LOADS], b_off[B_LOADS], corner[CONV ? A_LOADS : 1];
  // Which of B's loads a wave's i-th one is: where they do not divide among the waves, the last few are made twice.
  auto b_load = [&](int i) { return i * WAVES + wave - (i * WAVES + wave < B_BYTES / 1024 ? 0 : WAVES / 2); };
  constexpr int CHUNKS = STEP / 16, ROWS_PER_LOAD = 64 / CHUNKS, ROWS_PER_LINE = 256 / STEP;
  const int row16 = lane / CHUNKS, chunk = (lane % CHUNKS) ^ (row16 / ROWS_PER_LINE % CHUNKS);
  auto chunk_of = [&](int i) { return chunk ^ ((wave * A_LOADS + i) * ROWS_PER_LOAD / ROWS_PER_LINE % CHUNKS); };   // of A's i-th load
#pragma unroll
  for (int i = 0; i < A_LOADS; i++) {
    const int row = (wave * A_LOADS + i) * ROWS_PER_LOAD + row16;
    if constexpr (CONV) {   // its window's corner; rows past the last pixel are that one's again
      const uint32_t p = min(uint32_t(m0) + row, g.m - 1), line = g.conv.by_ow.div(p), img = g.conv.by_oh.div(line);
      corner[i] = ((img * g.conv.h + (line - img * g.conv.oh)) * g.conv.w + (p - line * g.conv.ow)) * g.conv.c_bytes + 4096 - i * 1024;
    } else {
      a_off[i] = uint32_t(row) * lda_b + chunk_of(i) * 16;
    }
  }
#pragma unroll
  for (int i = 0; i < B_LOADS; i++) {
    if constexpr (B_KMAJOR) b_off[i] = uint32_t((b_load(i)) * ROWS_PER_LOAD + row16) * ldb_b + (chunk ^ ((b_load(i)) * ROWS_PER_LOAD / ROWS_PER_LINE % CHUNKS)) * 16;
    else {
      constexpr int PITCH = BN * ES;
      const int at = (b_load(i)) * 1024 + lane * 16, r = at / PITCH;
      b_off[i] = uint32_t(r) * ldb_b + swizzle<T, BN>(at % PITCH, r);
    }
  }
  const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>((lds_void *)lds));
  // (what the loads' instruction offsets add, taken off 4096 bytes that the resources start earlier)
#pragma unroll
  for (int i = 0; i < A_LOADS && !CONV; i++) a_off[i] += 4096 - i * 1024;
#pragma unroll
  for (int i = 0; i < B_LOADS; i++) b_off[i] += 4096;
  // Where the step to request starts: the resources' bases.  Their sizes do not change from step to step (an offset past them is a
  // row's that does not exist), but for the steps that hold K's end and lie behind it.
  uint64_t a_tile = reinterpret_cast<uintptr_t>(A) - 4096, b_tile = reinterpret_cast<uintptr_t>(B) - 4096;
  uint32_t a_bytes = (CONV ? uint32_t(g.conv.image_bytes) : uint32_t(a_end)) + 4096, b_bytes = (B_KMAJOR ? b_end : b_rows(BK)) + 4096;
  int left = k_bytes;   // of K from the step to request on
  const uint32_t a_dst = lds0 + wave * (A_LOADS * 1024), b_dst = lds0 + A_BYTES;
  uint32_t fill = 0;   // the slot that it goes to
  const uint64_t b_step = B_KMAJOR ? uint64_t(STEP) : uint64_t(BK) * ldb_b;
  // Of the step that holds K's end, chunks past it become ones outside (the steps behind it are empty, so for good).
  auto end_of_k = [&]() __attribute__((always_inline)) {
    if (left <= 0) {
      a_bytes = b_bytes = 0;
      return;
    }
    if constexpr (!B_KMAJOR) b_bytes = b_rows(left / ES) + 4096;
    if constexpr (!CONV) each<A_LOADS>([&](auto i) { a_off[i] = chunk_of(i) * 16 >= left ? OUTSIDE : a_off[i]; });
    if constexpr (B_KMAJOR) each<B_LOADS>([&](auto i) { b_off[i] = (chunk ^ (b_load(i) * ROWS_PER_LOAD / ROWS_PER_LINE % CHUNKS)) * 16 >= left ? OUTSIDE : b_off[i]; });
  };
  // CONV: the window's byte that the step to request starts at, and where A's i-th chunk of that step lies.
  uint32_t window_byte = CONV ? blockIdx.y * g.conv.slice_bytes : 0;
  const uint32_t window_end = window_byte + k_bytes;
  auto find_chunk = [&](auto which) {
    constexpr int I = decltype(which)::value;
    const uint32_t kb = window_byte + chunk_of(I) * 16;
    a_off[I] = kb < window_end ? corner[I] + kb + g.conv.by_run.div(kb) * g.conv.run_gap : OUTSIDE;
    asm("" : "+v"(a_off[I]));   // here, and not behind the next barrier
  };
  constexpr int FINDS = CONV ? A_LOADS : 0;
  // Its i-th load of this wave.
  auto load = [&](auto which) {
    constexpr int I = decltype(which)::value;
    if constexpr (I < A_LOADS) dma16<I * 1024>(resource(a_tile, a_bytes), a_off[I], fill + a_dst);
    else dma16<0>(resource(b_tile, b_bytes), b_off[I - A_LOADS], fill + (b_dst + b_load(I - A_LOADS) * 1024));
  };
  auto next_slot = [&](uint32_t at) { return at + SLOT == SLOTS * SLOT ? 0u : at + SLOT; };
  // To the next step, in three parts.
  auto advance = [&](auto part) {
    constexpr int P = decltype(part)::value;
    if constexpr (P == 0) {
      left -= STEP;
      if constexpr (CONV) window_byte += STEP;
      else {
        a_tile += STEP;
        asm("" : "+s"(a_tile));   // (one sum a step, not an induction of the compiler's and three)
      }
    }
    if constexpr (P == 1) {
      b_tile += b_step;
      asm("" : "+s"(b_tile));
    }
    if constexpr (P == 2)
      if (left < STEP) end_of_k();
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
  v4i af[2][RA], bf[2][RB];
  // The addresses of a step's operands, in the slot `from`.
  const int a_rd = wm * WM * STEP + in_rows;
  constexpr int B_ADDRESSES = B_KMAJOR ? 1 : RB;
  if constexpr (B_KMAJOR) b_rd[0] = A_BYTES + wn * WN * STEP + in_rows;
  uint32_t a_at, b_at[B_ADDRESSES];
  auto locate = [&](uint32_t from, auto which) {
    constexpr int I = decltype(which)::value;
    uint32_t &at = I == 0 ? a_at : b_at[I == 0 ? 0 : I - 1];
    at = lds0 + from + (I == 0 ? a_rd : b_rd[I == 0 ? 0 : I - 1]);
    asm("" : "+v"(at));   // here, and not behind the barrier
  };
  // The i-th operand read of 64 bytes of K (RA of A, then RB of B).
  auto read = [&](auto set, auto which) {
    constexpr int S = decltype(set)::value, I = decltype(which)::value;
    if constexpr (I < RA) af[S][I] = *(lds_v4i *)uintptr_t(a_at + I * 16 * STEP);
    else if constexpr (B_KMAJOR) bf[S][I - RA] = *(lds_v4i *)uintptr_t(b_at[0] + (I - RA) * 16 * STEP);
    else {
      const uint8_t *at = (const uint8_t *)(lds_u8 *)uintptr_t(b_at[I - RA]);
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
  std::integral_constant<int, 0> even;
  std::integral_constant<int, 1> odd;
  // One MFMA after the other with a read or a load, if there are any to issue, behind it: what a wave
  // issues in one go its MFMAs wait for.  The last quarter has what the next step's reads and requests start from, so that no
  // arithmetic stands between the barrier and the first of either.
  auto step = [&](auto multiplied, auto fetched) {
    wait_for_all_but<(SLOTS - 2) * LOADS>();
    each<RA * RB>([&](auto q) {
      constexpr int Q = decltype(q)::value, N = RA * RB, READS = RA + RB, AHEAD = 3 + FINDS + 1 + B_ADDRESSES;
      multiply(multiplied, q);
      constexpr int R0 = min_of(READS, (Q * READS * 4 + N * 3 - 1) / (N * 3)), R1 = min_of(READS, ((Q + 1) * READS * 4 + N * 3 - 1) / (N * 3));   // in the first three quarters
      each<R1 - R0>([&](auto i) { read(fetched, std::integral_constant<int, R0 + decltype(i)::value>{}); });   // (behind the last step: zeros)
      constexpr int L0 = min_of(LOADS, Q * LOADS * 4 / (N * 3)), L1 = Q == N - 1 ? LOADS : min_of(LOADS, (Q + 1) * LOADS * 4 / (N * 3));
      each<L1 - L0>([&](auto i) { load(std::integral_constant<int, L0 + decltype(i)::value>{}); });
      constexpr int FROM = N - (N + 3) / 4, S0 = Q < FROM ? 0 : (Q - FROM) * AHEAD / (N - FROM), S1 = Q < FROM ? 0 : (Q + 1 - FROM) * AHEAD / (N - FROM);
      static_assert(N % 4 == 0 || N == 2, "the step's reads and loads are out by FROM");
      if constexpr (Q == FROM) fill = next_slot(fill);
      each<S1 - S0>([&](auto i) {
        constexpr int I = S0 + decltype(i)::value;
        if constexpr (I < 3) advance(std::integral_constant<int, I>{});
        else if constexpr (I < 3 + FINDS) find_chunk(std::integral_constant<int, I - 3>{});
        else locate(next_slot(fill), std::integral_constant<int, I - 3 - FINDS>{});
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  if (left < STEP) end_of_k();
  each<FINDS>([&](auto i) { find_chunk(i); });
#pragma unroll 1
  for (int s = 0; s < SLOTS; s++) {
    each<LOADS>([&](auto i) { load(i); });
    each<3>([&](auto i) { advance(i); });
    each<FINDS>([&](auto i) { find_chunk(i); });
    fill = next_slot(fill);
  }
  each<1 + B_ADDRESSES>([&](auto i) { locate(0, i); });
  wait_for_all_but<(SLOTS - 1) * LOADS>();
  each<RA + RB>([&](auto i) { read(even, i); });
  each<1 + B_ADDRESSES>([&](auto i) { locate(SLOT, i); });
  for (int k = 0; k + 2 <= steps; k += 2) {
    step(even, odd);
    step(odd, even);
  }
  if (steps & 1) each<RA * RB>([&](auto q) { multiply(even, q); });
  wait_for_all_but<0>();   // (requests past the last step write zeros)

  store_tile<T, A_UNSIGNED, RA, RB>(g, lds, acc, colsum, m0, n0, 0);
}

}  // namespace ring
}  // namespace mrl
