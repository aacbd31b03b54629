// Matmul tiles of 128 rows by 64 to 192 columns, and of 64 x 64, for problems that do not fill the chip with 256 x 256 ones: operands
// straight from memory into a ring of LDS slots of 128 bytes of K.
//
// What bounds a middling Matmul is less the MFMAs than everything around them: k_gemm's waves spend two
// thirds of a step issuing what is not an MFMA, in one go, or waiting for a step's trip through registers (bf16
// 1984 x 5120 x 1536, counters: MFMAs 33 % of the cycles), and tiles of 128 x 128 often come to a little over one per
// compute unit.  Here:
//   - operands go straight to LDS, and up to SLOTS steps are on their way at once.  Step k: wait until step
//     k + 1 has landed, barrier; then, dealt out between step k's MFMAs, the reads of step k + 1's operands and the
//     requests of step k + SLOTS, into the slot that step k's operands were read from (they are in registers
//     before the barrier);
//   - eight waves: four blocks of 64 x BN / 2 outputs, each once for the first and once for the second 64 bytes of
//     every step, whose sums meet in LDS at the end: two waves on a SIMD, one issuing while the other's MFMAs
//     run, and an operand read still serves BN / 32 or four MFMAs;
//   - widths chosen so that the tiles fill one round (gemm_ring_columns);
//   - nothing but the barrier between a step's last MFMA and the next one's first: what the next step's reads and requests start from
//     is worked out behind the MFMAs of the step before.  (Some 35 scalar instructions in one go behind the last MFMA, while both waves of a SIMD had
//     none under way: bf16 2048^3 22.0 us, now 21.0, u8 1472 x 2304 x 2752 21.0 / 19.2, 1546 x 5000 x 2560 41.3 / 37.8.)
// What bounds the loop now is the way into LDS: a step of the 128 x 128 tile takes 0.36 us, its loads by themselves 0.31 (105 bytes a
// nanosecond and unit), its MFMAs 0.21.
// The loads are buffer loads: rows past M or N and chunks past K come as zeros, without a branch.
//
// LDS: A as [row][128 bytes], 16-byte chunks XOR-ed with (row / 2) & 7; a k-fastest B likewise; a
// row-major B as [k][columns], the pieces that transposing reads take (16 columns) XOR-ed so that the
// rows that one half of a wave reads at once lie in different banks.  Loads fill LDS in order, so
// the swizzles are applied to the addresses in memory.
// Semantics: morello/src/spec.rs:480-485; integers exact, bf16 summed in f32.
#include "gemm_ring.h"

namespace mrl {
namespace {
using namespace ring;
using gemm::TileWalk;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) const uint8_t lds_u8;
typedef __attribute__((address_space(3))) const v4i lds_v4i;

constexpr uint32_t OUTSIDE = 0x80000000u;   // an offset no resource here holds

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

template <class T, bool A_UNSIGNED, bool B_KMAJOR, int RA, int RB, int SLOTS>
__global__ __launch_bounds__(64 * WAVES, RB <= 2 ? 4 : 2) void k_gemm_ring(MRL_WALK_PARAMS, GemmArgs g) {
  typedef typename Ring<T>::Acc Acc;
  constexpr int ES = T::ES, BK = STEP / ES, BM = 32 * RA, BN = 32 * RB, WM = 16 * RA, WN = 16 * RB;
  constexpr int A_BYTES = BM * STEP, B_BYTES = BN * STEP, SLOT = A_BYTES + B_BYTES;
  constexpr int A_LOADS = A_BYTES / (1024 * WAVES), B_LOADS = (B_BYTES / 1024 + WAVES - 1) / WAVES, LOADS = A_LOADS + B_LOADS;   // a wave's, per step
  static_assert((SLOTS - 1) * LOADS < 64 && A_LOADS <= 4 && B_LOADS <= 4, "");
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kw = wave >> 2, wm = wave >> 1 & 1, wn = wave & 1;
  MRL_WALK_TILE(tile_m, tile_n)
  const int64_t m0 = int64_t(tile_m) * BM, n0 = int64_t(tile_n) * BN;
  const uint8_t *A = (const uint8_t *)g.a + (int64_t(blockIdx.y) * g.sa + m0 * g.lda) * ES;
  const bool panels = !B_KMAJOR && g.b_panel_rows != 0;
  const uint8_t *B = (const uint8_t *)g.b + (int64_t(blockIdx.y) * g.sb + (B_KMAJOR ? n0 * g.ldb : panels ? n0 * g.b_panel_rows : n0)) * ES;
  const uint32_t lda_b = uint32_t(g.lda) * ES, ldb_b = panels ? BN * ES : uint32_t(g.ldb) * ES;
  // Bytes of the tile's rows (leading dimensions stay below 2^24 bytes); what of a row-major B's lies left of the tile.
  const int a_end = min(BM, int(g.m - m0)) * int(lda_b), n0_b = panels ? 0 : int(n0) * ES;
  const uint32_t b_end = uint32_t(min(BN, int(g.n - n0))) * ldb_b;
  const int k = g.k_total != 0 ? int(min(g.k, g.k_total - blockIdx.y * g.k)) : int(g.k), k_bytes = k * ES, steps = (k_bytes + STEP - 1) / STEP;

  // Where this lane's chunks of a step come from.  Rows of 64 bytes: sixteen to a load.
  uint32_t a_off[A_LOADS], b_off[B_LOADS];
  // Which of B's loads a wave's i-th one is: where they do not divide among the waves, the last few are made twice.
  auto b_load = [&](int i) { return i * WAVES + wave - (i * WAVES + wave < B_BYTES / 1024 ? 0 : WAVES / 2); };
  constexpr int CHUNKS = STEP / 16, ROWS_PER_LOAD = 64 / CHUNKS, ROWS_PER_LINE = 256 / STEP;
  const int row16 = lane / CHUNKS, chunk = (lane % CHUNKS) ^ (row16 / ROWS_PER_LINE % CHUNKS);
#pragma unroll
  for (int i = 0; i < A_LOADS; i++) a_off[i] = uint32_t((wave * A_LOADS + i) * ROWS_PER_LOAD + row16) * lda_b + (chunk ^ ((wave * A_LOADS + i) * ROWS_PER_LOAD / ROWS_PER_LINE % CHUNKS)) * 16;
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
  for (int i = 0; i < A_LOADS; i++) a_off[i] += 4096 - i * 1024;
#pragma unroll
  for (int i = 0; i < B_LOADS; i++) b_off[i] += 4096;
  // Where the step to request starts: the resources' bases.  Their sizes do not change from step to step (an offset past them is a
  // row's that does not exist), but for the steps that hold K's end and lie behind it.
  uint64_t a_tile = reinterpret_cast<uintptr_t>(A) - 4096, b_tile = reinterpret_cast<uintptr_t>(B) - 4096;
  uint32_t a_bytes = uint32_t(a_end) + 4096, b_bytes = (B_KMAJOR ? b_end : uint32_t(BK) * ldb_b - n0_b) + 4096;
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
    if constexpr (!B_KMAJOR) b_bytes = uint32_t(left / ES) * ldb_b - n0_b + 4096;
    each<A_LOADS>([&](auto i) { a_off[i] = (chunk ^ ((wave * A_LOADS + i) * ROWS_PER_LOAD / ROWS_PER_LINE % CHUNKS)) * 16 >= left ? OUTSIDE : a_off[i]; });
    if constexpr (B_KMAJOR) each<B_LOADS>([&](auto i) { b_off[i] = (chunk ^ (b_load(i) * ROWS_PER_LOAD / ROWS_PER_LINE % CHUNKS)) * 16 >= left ? OUTSIDE : b_off[i]; });
  };
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
      a_tile += STEP, left -= STEP;
      asm("" : "+s"(a_tile));   // (one sum a step, not an induction of the compiler's and three)
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
      constexpr int Q = decltype(q)::value, N = RA * RB, READS = RA + RB, AHEAD = 3 + 1 + B_ADDRESSES;
      multiply(multiplied, q);
      constexpr int R0 = min_of(READS, (Q * READS * 4 + N * 3 - 1) / (N * 3)), R1 = min_of(READS, ((Q + 1) * READS * 4 + N * 3 - 1) / (N * 3));   // in the first three quarters
      each<R1 - R0>([&](auto i) { read(fetched, std::integral_constant<int, R0 + decltype(i)::value>{}); });   // (behind the last step: zeros)
      constexpr int L0 = min_of(LOADS, Q * LOADS * 4 / (N * 3)), L1 = Q == N - 1 ? LOADS : min_of(LOADS, (Q + 1) * LOADS * 4 / (N * 3));
      each<L1 - L0>([&](auto i) { load(std::integral_constant<int, L0 + decltype(i)::value>{}); });
      constexpr int FROM = N - (N + 3) / 4, S0 = Q < FROM ? 0 : (Q - FROM) * AHEAD / (N - FROM), S1 = Q < FROM ? 0 : (Q + 1 - FROM) * AHEAD / (N - FROM);
      static_assert(N % 4 == 0, "the step's reads and loads are out by FROM");
      if constexpr (Q == FROM) fill = next_slot(fill);
      each<S1 - S0>([&](auto i) {
        constexpr int I = S0 + decltype(i)::value;
        if constexpr (I < 3) advance(std::integral_constant<int, I>{});
        else locate(next_slot(fill), std::integral_constant<int, I - 3>{});
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto advance_whole = [&]() { each<3>([&](auto i) { advance(i); }); };
  if (left < STEP) end_of_k();
#pragma unroll 1
  for (int s = 0; s < SLOTS; s++) {
    each<LOADS>([&](auto i) { load(i); });
    advance_whole();
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

template <class T, bool A_UNSIGNED, bool B_KMAJOR, int RA, int RB, int SLOTS>
hipError_t launch_ring(const GemmArgs &g, hipStream_t stream) {
  constexpr auto kern = k_gemm_ring<T, A_UNSIGNED, B_KMAJOR, RA, RB, SLOTS>;
  constexpr int BM = 32 * RA, BN = 32 * RB, LDS = SLOTS * (BM + BN) * STEP;
  static_assert(LDS >= 4 * 16 * RA * (16 * RB + 4) * 4, "the waves' pieces of C fit");
  static std::atomic<uint64_t> lds_limit_set{0};
  if (!plan::recording() && LDS > 65536) {
    hipError_t e = raise_lds_limit(lds_limit_set, (const void *)kern, LDS);
    if (e != hipSuccess) return e;
  }
  const int tiles_m = int((g.m + BM - 1) / BM), tiles_n = int((g.n + BN - 1) / BN);
  const double mn = double(g.m) * g.n * g.batch, steps = double((uint64_t(g.k) * T::ES + STEP - 1) / STEP);
  plan::work(T::ES == 1 ? plan::UNIT_MFMA_I8 : plan::UNIT_MFMA_BF16, 2.0 * mn * g.k,
             (double(g.m) * g.k + double(g.k) * g.n) * g.batch * T::ES + mn * (g.c_bf16 ? 2 : 4) * (g.accum ? 2 : 1),
             2.0 * BM * BN * steps * (STEP / T::ES), 2500.0 + 300.0 * steps);
  const TileWalk walk = gemm::tile_walk(tiles_m, tiles_n);
  MRL_LAUNCH((k_gemm_ring<T, A_UNSIGNED, B_KMAJOR, RA, RB, SLOTS>), dim3(tiles_m * tiles_n, g.batch), dim3(64 * WAVES), LDS, stream, MRL_WALK_ARGS(walk), g);
  return plan::last_error();
}

template <class T, bool A_UNSIGNED, int RA, int RB, int SLOTS>
hipError_t launch_either(const GemmArgs &g, hipStream_t stream) {
  return g.b_kmajor ? launch_ring<T, A_UNSIGNED, true, RA, RB, SLOTS>(g, stream) : launch_ring<T, A_UNSIGNED, false, RA, RB, SLOTS>(g, stream);
}
// As many slots as a compute unit's LDS holds of the wider ones, and four of the 64-wide tile's as well: all run one to a unit (of the
// last, three / four / six: bf16 1024 x 7040 x 1344 35.7 / 33.2 / 33.4 us, 1664 x 6720 x 1152 34.6 / 33.0 / 33.2; of 128, five instead of four are within 1 %).  Four of the 64 x 64
// tile, two of which share a unit (us, three / four / six / eight: bf16 192 x 768 x 384 4.74 / 4.81 / 4.9 / 5.2, 313 x 2176 x 267 twice 10.7 / 9.3 / 9.2 /
// 9.5, u8 600 x 2496 x 236 7.3 / 7.3 / 7.6 / 7.9, 693 x 4352 x 817 11.9 / 10.8).
template <class T, bool A_UNSIGNED>
hipError_t launch_kind(const GemmArgs &g, uint32_t bn, hipStream_t stream) {
  switch (bn) {
    case 32: return launch_either<T, A_UNSIGNED, 2, 2, 4>(g, stream);
    case 64: return launch_either<T, A_UNSIGNED, 4, 2, 4>(g, stream);
    case 128: return launch_either<T, A_UNSIGNED, 4, 4, 4>(g, stream);
    case 160: return launch_either<T, A_UNSIGNED, 4, 5, 4>(g, stream);
    case 192: return launch_either<T, A_UNSIGNED, 4, 6, 4>(g, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

// Measured against k_gemm's tiles (us, k_gemm / this; means of 520 random sizes, of three sets of operands in turn), on rounds of one
// tile per compute unit:
//   64 where k_gemm's 64 tile would go two to a unit (257 of them on) and this one at most one: bf16 1100 x 3001 x
//     1100 35.1 / 28.0, u8 1408 x 3001 x 1408 23.6 / 20.9; two to a unit it loses (400 x 3001 x 4400 35.7 / 46.4).  bf16 from 13
//     steps on (13 to 15 1.13 times as fast, 1.11 with operands from memory; 11 and 12 1.05 and from memory 0.85 at the least, nine and ten 1.02 and
//     0.91), integers from 14 (14 to 16 1.11, from memory 1.09; 11 to 13 1.04 and 0.97, seven and eight 0.98);
//   128 for more than half a round of 128 x 128.  Integers from 28 steps on: 4054 x 4352 x 832 26.6 / 24.1 (28 and 29 1.07, 30 to 34 1.06, from memory
//     1.03; 23 to 25 1.02 and from memory 0.97, 11 to 16 0.94).  bf16 too: 2048^3 22.9 / 22.2 (28 and 29 1.04, 30 to 34 1.09, from memory 1.07;
//     23 to 26 1.06, but 0.93 for one in six; 9 to 16 0.95).  Where 64 x 64 tiles are 512 at most, which k_gemm runs two to a unit, both from 36
//     (integers 35 to 44 1.08, bf16 45 on 1.22; 30 to 34 1.02 and from memory 0.95, 11 to 19 0.89);
//   160, else 192, where the 128 tile needs a second round and they do not: bf16 1001 x 2050 x 4425 47.2 / 38.9, 1800 x 2001
//     x 3000 41.0 / 35.3, u8 1000 x 2001 x 4500 34.6 / 30.1.  (128 in two rounds: 0.92 to 1.03, and 0.90 with operands from memory.)
// Short K leaves the start of the ring and the summing of the two halves of K dominant: bf16 1408 x 320 x 1408 5.9 / 6.7.
uint32_t gemm_ring_columns(const GemmArgs &g, int kind) {
  if (kind < 0 || kind > 2) return 0;
  const uint64_t es = kind == 2 ? 2 : 1, steps = (uint64_t(g.k) * es + STEP - 1) / STEP;
  auto tiles = [&](uint32_t bm, uint32_t bn) { return uint64_t((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * g.batch; };
  const uint64_t units = g_compute_units, small = tiles(64, 64), whole = tiles(128, 128);
  if (steps < (kind == 2 ? 13 : 14) || g.m <= 128 || g.n <= 128) return 0;
  if (small <= 512) {
    if (small <= units) return 0;
    return tiles(128, 64) <= units ? 64 : 2 * whole > units && steps >= 36 ? 128 : 0;
  }
  if (whole <= units) return 2 * whole > units && steps >= 28 ? 128 : 0;
  if (steps < 16) return 0;
  return tiles(128, 160) <= units ? 160 : tiles(128, 192) <= units ? 192 : 0;
}

hipError_t launch_gemm_ring(const GemmArgs &g, int kind, uint32_t bn, hipStream_t stream) {
  switch (kind) {
    case 0: return launch_kind<I8, false>(g, bn, stream);
    case 1: return launch_kind<I8, true>(g, bn, stream);
    case 2: return launch_kind<BF16, false>(g, bn, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mrl
