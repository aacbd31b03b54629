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
#include "gemm_ring_tile.h"

namespace mrl {
namespace {
using namespace ring;
using gemm::TileWalk;
template <class T, bool A_UNSIGNED, bool B_KMAJOR, int RA, int RB, int SLOTS>
__global__ __launch_bounds__(64 * WAVES, RB <= 2 ? 4 : 2) void k_gemm_ring(MRL_WALK_PARAMS, GemmArgs g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  MRL_WALK_TILE(tile_m, tile_n)
  ring_tile<T, A_UNSIGNED, B_KMAJOR, RA, RB, SLOTS>(lds, tile_m, tile_n, g);
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
             2.0 * BM * BN * steps * (STEP / T::ES), RA * RB > 4 ? 2500.0 + 300.0 * steps : 900.0 + (B_KMAJOR ? (T::ES == 2 ? 155.0 : 185.0) : T::ES == 2 ? 220.0 : 275.0) * steps);
  const TileWalk walk = gemm::tile_walk(tiles_m, tiles_n);
  MRL_LAUNCH((k_gemm_ring<T, A_UNSIGNED, B_KMAJOR, RA, RB, SLOTS>), dim3(tiles_m * tiles_n, g.batch), dim3(64 * WAVES), LDS, stream, MRL_WALK_ARGS(walk), g);
  return plan::last_error();
}

template <class T, bool A_UNSIGNED, int RA, int RB, int SLOTS>
hipError_t launch_either(const GemmArgs &g, hipStream_t stream) {
  return g.b_kmajor ? launch_ring<T, A_UNSIGNED, true, RA, RB, SLOTS>(g, stream) : launch_ring<T, A_UNSIGNED, false, RA, RB, SLOTS>(g, stream);
}
// As many slots as a compute unit's LDS holds of the wider ones, and four of the 64-wide tile's as well: all run one
// to a unit (of the last, three / four / six: bf16 1024 x 7040 x 1344 35.7 / 33.2 / 33.4 us, 1664 x 6720 x 1152 34.6
// / 33.0 / 33.2; of 128, five instead of four are within 1 %).  Four of the 64 x 64 tile, two of which share a unit
// (us, three / four / six / eight: bf16 192 x 768 x 384 4.74 / 4.81 / 4.9 / 5.2, 313 x 2176 x 267 twice 10.7 / 9.3 /
// 9.2 / 9.5, u8 600 x 2496 x 236 7.3 / 7.3 / 7.6 / 7.9, 693 x 4352 x 817 with a k-fastest B 11.9 / 10.8).
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

// Measured against k_gemm's tiles (us, k_gemm / this; means of 520 random sizes, of three sets of operands in turn),
// on rounds of one tile per compute unit:
//   64 where k_gemm's 64 tile would go two to a unit (257 of them on) and this one at most one: bf16 1100 x 3001 x
//     1100 35.1 / 28.0, u8 1408 x 3001 x 1408 23.6 / 20.9; two to a unit it loses (400 x 3001 x 4400 35.7 / 46.4).
//     bf16 from 13 steps on, integers from 14 (335 sizes up to 15, one set of operands / three in turn / B from
//     memory / all of it: rows of whole cache lines 1.23 / 1.11 / 1.11 / 1.04, others of a k-fastest B 1.16 / 1.04 /
//     1.04 / 0.97, of a row-major one 1.11 / 1.02 / 1.00 / 0.93; bf16 of 11 and 12 1.05 and from memory 0.85 at the
//     least, integers of 11 to 13 1.04 and 0.97);
//   128 for more than half a round of 128 x 128.  Integers from 28 steps on: 4054 x 4352 x 832 26.6 / 24.1 (28 and 29
//     1.07, 30 to 34 1.06, from memory 1.03; 23 to 25 1.02 and from memory 0.97, 11 to 16 0.94).  bf16 too: 2048^3
//     22.9 / 22.2 (28 and 29 1.04, 30 to 34 1.09, from memory 1.07; 23 to 26 1.06, but 0.93 for one in six; 9 to 16
//     0.95).  Where 64 x 64 tiles are 512 at most, which k_gemm runs two to a unit, both from 36 (integers 35 to 44
//     1.08, bf16 45 on 1.22; 30 to 34 1.02 and from memory 0.95, 11 to 19 0.89);
//   160, else 192, where the 128 tile needs a second round and they do not: bf16 1001 x 2050 x 4425 47.2 / 38.9, 1800
//     x 2001 x 3000 41.0 / 35.3, u8 1000 x 2001 x 4500 34.6 / 30.1.  (128 in two rounds: 0.92 to 1.03, and 0.90 with
//     operands from memory.)
// Rows of K that are no whole cache lines, of which a step's 128 bytes lie in two, cost the 128-wide tile that much
// more than k_gemm's: i8 from 60 steps on, a k-fastest bf16 B from 32, and where 64 x 64 tiles are 512 at most a
// k-fastest B of either not at all (one set of operands / three in turn / B from memory / all of it, means: i8 below
// 60 0.97 / 0.96 / 0.96 / 0.93, from there 1.02 / 1.01 / 1.00 / 0.96, of whole lines 1.09 / 1.09 / 1.04 / 0.99; bf16
// 0.93 / 0.94 / 0.94 / 0.92, of whole lines 1.09 / 1.09 / 1.04 / 1.00; i8 883 x 4928 x 2336 26.0 / 27.0, twice 792 x
// 3552 x 1760 21.7 / 24.6, bf16 twice 1109 x 1768 x 1504 21.1 / 23.5).  u8 pays k_gemm for its columns' sums (1.04 /
// 1.04 / 1.03 / 1.00).  Where 128 x 128 pads much more than 64 x 64 the other choice is k_gemm's 64 tile, 1.8 times
// as slow.
// Short K leaves the start of the ring and the summing of the two halves of K dominant: bf16 1408 x 320 x 1408 5.9 /
// 6.7.
uint32_t gemm_ring_columns(const GemmArgs &g, int kind) {
  if (kind < 0 || kind > 2) return 0;
  const uint64_t es = kind == 2 ? 2 : 1, steps = (uint64_t(g.k) * es + STEP - 1) / STEP;
  auto tiles = [&](uint32_t bm, uint32_t bn) { return uint64_t((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * g.batch; };
  const uint64_t units = g_compute_units, small = tiles(64, 64), whole = tiles(128, 128);
  if (steps < (kind == 2 ? 13 : 14) || g.m <= 128 || g.n <= 128) return 0;
  const bool k_lines = g.lda * es % STEP == 0;
  if (small <= 512) {
    if (small <= units) return 0;
    if (tiles(128, 64) <= units) return 64;
    return 2 * whole > units && steps >= 36 && (k_lines || !g.b_kmajor || kind == 1) ? 128 : 0;
  }
  if (whole <= units) {
    // (i8 of other rows stays for a whole round, whose route tests/test_gpu_matmul_ring_widths.py holds fast for 2048
    // x 3472 x 2048, 21.4 / 22.5)
    const bool as_lines = k_lines || gemm_tile_side(g, kind) == 64 || (kind == 0 ? whole == units : kind == 1 || !g.b_kmajor);
    return 2 * whole > units && steps >= (as_lines ? 28 : kind == 2 ? 32 : 60) ? 128 : 0;
  }
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
