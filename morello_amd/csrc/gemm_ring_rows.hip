// The tiles of gemm_ring.hip for operands whose rows start anywhere: K or N not a multiple of 16 bytes, operands read
// where they lie.
//
// The other tiled kernels want rows of whole 16-byte chunks and get them from padded copies: a launch and a pass over
// both operands, a third to a half of a small ragged Matmul's time (over 350 random sizes that the rule below takes,
// the geometric mean against that is 0.73).  Here the chunks are loads of 16 bytes at any address, through registers
// into LDS (a load straight to LDS has to be aligned):
//   - step k: barrier; then, dealt out between its MFMAs, the reads of step k + 1's operands, the writes of step k +
//     2's chunks into the slot that step k's operands were read from, and the loads of step k + 2 + DEPTH into the
//     registers these leave.  Two slots of LDS, DEPTH steps of loads under way;
//   - the first step takes what K has over whole steps, zeros behind it, so that the k loop has no remainder: its
//     chunks are whole, and inside their rows;
//   - rows past M (or N) are the last one again, and a row-major B's last tile starts BN columns before B's end and
//     leaves those its neighbour has: no load leaves the operands, and none is masked but the first step's.
// What bounds it is the step's chain of barrier, operand reads and MFMAs, 0.25 to 0.33 us on the smallest tile
// (k_gemm's step: 0.4 to 0.5; gemm_ring.hip's, of whole chunks, 0.17 to 0.2), and past one workgroup a unit the cache
// lines that unaligned rows touch twice. Everything else as in gemm_ring.hip. Semantics: morello/src/spec.rs:480-485;
// integers exact, bf16 summed in f32.
#include "gemm_ring_rows.h"

namespace mrl {
namespace {
using namespace ring;
using gemm::TileWalk;
template <class T, bool A_UNSIGNED, bool B_KMAJOR, int RA, int RB>
__global__ __launch_bounds__(64 * WAVES, RA * RB <= 4 ? 4 : 2) void k_gemm_ring(MRL_WALK_PARAMS, GemmArgs g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  MRL_WALK_TILE(tile_m, tile_n)
  rows_tile<T, A_UNSIGNED, B_KMAJOR, RA, RB>(lds, tile_m, tile_n, g);
}

template <class T, bool A_UNSIGNED, bool B_KMAJOR, int RA, int RB>
hipError_t launch_rows(const GemmArgs &g, hipStream_t stream) {
  constexpr auto kern = k_gemm_ring<T, A_UNSIGNED, B_KMAJOR, RA, RB>;
  constexpr int BM = 32 * RA, BN = 32 * RB, LDS = std::max(2 * (BM + BN) * STEP, 4 * 16 * RA * (16 * RB + 4) * 4);
  if (g.m < 1 || (!B_KMAJOR && g.n < uint32_t(BN)) || uint64_t(g.k) * T::ES <= STEP) return hipErrorInvalidValue;
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
  MRL_LAUNCH((k_gemm_ring<T, A_UNSIGNED, B_KMAJOR, RA, RB>), dim3(tiles_m * tiles_n, g.batch), dim3(64 * WAVES), LDS, stream, MRL_WALK_ARGS(walk), g);
  return plan::last_error();
}

template <class T, bool A_UNSIGNED, int RA, int RB>
hipError_t launch_either(const GemmArgs &g, hipStream_t stream) {
  return g.b_kmajor ? launch_rows<T, A_UNSIGNED, true, RA, RB>(g, stream) : launch_rows<T, A_UNSIGNED, false, RA, RB>(g, stream);
}
template <class T, bool A_UNSIGNED>
hipError_t launch_kind(const GemmArgs &g, uint32_t bn, hipStream_t stream) {
  switch (bn) {
    case 32: return launch_either<T, A_UNSIGNED, 2, 2>(g, stream);
    case 64: return launch_either<T, A_UNSIGNED, 4, 2>(g, stream);
    case 128: return launch_either<T, A_UNSIGNED, 4, 4>(g, stream);
    case 160: return launch_either<T, A_UNSIGNED, 4, 5>(g, stream);
    case 192: return launch_either<T, A_UNSIGNED, 4, 6>(g, stream);
    default: return hipErrorInvalidValue;
  }
}

// More than half of a round of 64 x 64 tiles and up to three quarters: K is not shared out here (a second round), and
// k_gemm's slices of it, three workgroups to a unit, are the faster way over a long K where they come cheap (us,
// those / this, bf16 where not said):
//   no operand to copy, from 61 steps on, those whose K is whole chunks as well against the tile of gemm_ring.hip,
//     which has them now: 678 x 5488 x 755 23.8 / 27.9, 1086 x 3848 x 533 21.2 / 21.7, 492 x 4664 x 1414 24.1 / 26.2,
//     u8 201 x 10320 x 2955 25.8 / 29.0 (where the line was drawn: 59 steps 20.1 / 21.1; 231 x 3872 x 3091, 196
//     tiles, 23.2 / 22.1);
//   K, ending on a whole chunk, in three equal slices or more: 653 x 5434 x 782 24.6 / 31.2, 460 x 4031 x 1299 23.0 /
//     26.6;
//   only B to copy, from 77 steps on: 755 x 4992 x 741 22.7 / 26.8, 1775 x 5520 x 268 27.3 / 29.1 (1415 x 4448 x 443
//     26.9 / 24.5);
//   int8 rows of N, of which a step takes half lines, from 67 steps on: 905 x 9285 x 519 29.7 / 35.7.
// Other ragged ones are faster here: 1150 x 4530 x 497 28.1 / 26.5, 265 x 4822 x 2236 34.0 / 29.9.
bool slices_are_faster(const GemmArgs &g, int kind, int es, uint64_t steps, uint64_t small, uint64_t units) {
  if (4 * small > 3 * units || steps <= 60) return false;
  const int64_t chunk = 16 / es;
  const bool a_whole = g.lda % chunk == 0, b_whole = g.ldb % chunk == 0;
  if (a_whole && b_whole) return true;
  GemmArgs copied = g;
  copied.k = uint32_t((g.k + chunk - 1) / chunk * chunk);
  uint32_t left = 0;
  if (gemm_k_splits(copied, kind, &left) >= 3 && left == 0) return true;
  const bool few_tiles = 8 * small <= 5 * units;
  return few_tiles && ((steps > 76 && a_whole && uint64_t(g.n) * g.k * es <= (11u << 20)) || (steps > 66 && kind <= 1 && !g.b_kmajor));
}
// 33 to 64 rows of whole chunks, which k_gemm reads in place too.  Its slices were the faster way, against the tile
// here, for the sizes below.  gemm_ring.hip's tile has those that stay now, and the lines have not been drawn again
// for it (us, k_gemm's slices / that tile, three sets of operands in turn, all of it from memory):
//   three equal slices or more against 30 MB of B or more: bf16 47 x 8192 x 5696 23.8 / 27.1, 25.8 / 29.3, 56 x 4480
//     x 9721 22.5 / 23.9, 25.5 / 27.9, 33 x 3456 x 14243 25.4 / 22.0, 26.4 / 23.1, 52 x 7040 x 2911 13.4 / 13.3, 15.3
//     / 15.3, u8 41 x 10240 x 10752 30.5 / 30.4, 30.6 / 30.7, 45 x 3840 x 8607 12.1 / 10.4, 15.4 / 14.6;
//   with one left over, from 129 tiles to seven tenths of a round past 60 steps: u8 40 x 10496 x 8431 26.1 / 25.2,
//     29.2 / 29.1, bf16 45 x 3904 x 8991 20.2 / 14.7, 25.2 / 23.1; of whole steps, to five eighths past 52 as well,
//     and past 110 steps and ten thousand of all tiles: 35 x 8768 x 5888 28.6 / 28.2, 29.2 / 28.6, 39 x 11712 x 4800
//     32.0 / 27.3, 32.2 / 27.5.
bool slices_are_faster_of_few(const GemmArgs &g, int kind, int es, uint64_t steps, uint64_t small, uint64_t units) {
  const int64_t chunk = 16 / es;
  if (g.lda % chunk != 0 || g.ldb % chunk != 0 || g.k % chunk != 0) return false;
  uint32_t left = 0;
  const uint32_t slices = gemm_k_splits(g, kind, &left);
  if (left == 0) return slices >= 3 && uint64_t(g.n) * g.k * es >= 30000000;
  if (2 * small > units && steps > 60) return 10 * small <= 7 * units;
  if (uint64_t(g.k) * es % STEP != 0) return false;
  return 2 * small > units ? steps > 52 && 8 * small <= 5 * units : steps > 110 && small * steps > 10000;
}

}  // namespace

// Measured against padded copies and the kernels of gemm_mfma.hip (us, those / this):
//   32 (64 x 64) where such tiles are one round at most: bf16 613 x 2516 x 936 24.5 / 15.7, 907 x 1546 x 235 twice
//     20.5 / 11.5, 2033 x 340 x 350 8.6 / 5.1, 796 x 4509 x 96 in slices of K 22.6 / 10.0, u8 1015 x 2999 x 803 20.9
//     / 15.0, 1000^3, exactly a round, 10.4 / 7.4, 1060 x 10040 x 103 25.7 / 11.6, 300 x 270 x 290 6.7 / 4.4;
//   64 (128 x 64) where those are: bf16 975 x 2176 x 1666 22.5 / 17.5, u8 1888 x 1633 x 885 17.4 / 14.7; int8 over a
//     long K reads its rows' lines once too often: 1651 x 5949 x 844 28.8 / 31.8, and bf16 over a longer one: 1835 x
//     3535 x 655 31.7 / 35.2;
//   128 (128 x 128), bf16: 1483 x 858 x 1983 18.4 / 15.8, 1303 x 1524 x 2056 24.3 / 20.3; over a long K the copies
//     are the faster way (1538 x 3021 x 1767 34.2 / 38.6), for int8 rows of an odd number of bytes at once (1055 x
//     929 x 1801 13.2 / 15.8); k-fastest B of others 875 x 3964 x 2980 35.0 / 25.9, 726 x 996 x 4035 17.8 / 13.6;
//   160 (128 x 160) where those are and 128 x 128 ones are not, else 192 (128 x 192), bf16: 2306 x 735 x 2260 24.5 /
//     17.4, 2491 x 1862 x 2026 38.8 / 31.3, k-fastest B twice 771 x 813 x 3032 29.1 / 21.2; u8 2078 x 1500 x 2672
//     28.4 / 21.6.
uint32_t gemm_ring_rows_columns(const GemmArgs &g, int kind) {
  if (kind < 0 || kind > 2) return 0;
  const int es = kind == 2 ? 2 : 1;
  const uint64_t steps = (uint64_t(g.k) * es + STEP - 1) / STEP;
  // More than 32 rows against a large k-fastest B: half a tile or more, and K in slices fills the chip where gemm_skinny.hip
  // and k_gemm have a workgroup for 16, 32 or 64 columns (bf16 38 x 10482 x 1472 24.0 / 11.7, 57 x 1856 x 4284 13.4 / 9.6, u8 41 x
  // 6895 x 2728 17.3 / 11.5; below 10 MB of B they are the faster ones: u8 39 x 3840 x 1920 6.2 / 8.6).
  const bool few = g.m <= 64;
  if (few && !(g.m > 32 && g.b_kmajor && g.batch == 1 && uint64_t(g.n) * g.k * es > (10ull << 20))) return 0;
  if (g.n <= 64 || steps < 2 || steps >= (1u << 22) || !gemm::edge_addressable(g, es) || g.batch > 65535 ||
      reinterpret_cast<uintptr_t>(g.c) % (g.c_bf16 ? 2 : 4) != 0)
    return 0;
  auto tiles = [&](uint32_t bm, uint32_t bn) { return uint64_t((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * g.batch; };
  const uint64_t units = g_compute_units, small = tiles(64, 64);
  if (g.tight)   // no scratch for copies or partial results, whatever it costs
    return small <= units ? 32 : tiles(128, 64) <= units ? 64 : kind == 2 && g.n >= 128 && tiles(128, 128) <= units ? 128 : 0;
  // bf16 rows of an odd number of elements along K, a pair of lines for every 128 bytes of either operand: most where
  // the operands come from memory (us, those / this, from memory and with three sets of operands in turn, which the
  // memory-side cache keeps).
  const bool odd_rows = kind == 2 && g.b_kmajor && (g.lda % 2 != 0 || g.ldb % 2 != 0);
  if (small <= units) {
    if (few && slices_are_faster_of_few(g, kind, es, steps, small, units)) return 0;
    // Half a round of tiles whose K is too short to share out: 43 x 1273 x 4452 11.5 / 14.8, 9.4 / 10.6, 49 x 1043 x
    // 7166 12.0 / 13.6, 9.9 / 10.0 (of words 43 x 1084 x 5269 11.0 / 12.1, 9.1 / 8.4; 35 x 971 x 8647, 136 tiles,
    // 19.3 / 13.2, 16.8 / 10.4; 39 x 1603 x 3436, 26 steps in three, 13.0 / 11.2, 10.3 / 10.1).
    if (few && odd_rows && 2 * small <= units && steps < 24) return 0;
    if (2 * small <= units) return 32;
    if (steps > 88) return 0;   // (292 x 6007 x 2192 bf16, 175 tiles of 94 steps: 34.7 / 35.8)
    return g.batch == 1 && !few && slices_are_faster(g, kind, es, steps, small, units) ? 0 : 32;
  }
  // In one entry from 41 steps on (1031 x 2937 x 1194 26.7 / 32.0, 407 x 2585 x 2924 24.4 / 26.9; 231 x 2739 x 4310
  // 27.5 / 26.5, 2270 x 2473 x 710 26.5 / 24.5), in several from 31 (twice 581 x 2761 x 1178 28.5 / 37.2, 27.0 /
  // 29.4, 887 x 1961 x 904 24.6 / 28.3, 22.7 / 21.6; 1343 x 1481 x 639 24.6 / 25.5, 22.4 / 19.3).
  if (tiles(128, 64) <= units) return steps <= (kind != 2 ? 24u : !odd_rows ? 48u : g.batch == 1 ? 40u : 30u) ? 64 : 0;
  // Of 128 x 128 up to two thirds of a round from 16 (twice 789 x 1007 x 1167 20.9 / 25.1, 19.0 / 21.1, 2399 x 1307
  // x 925 25.3 / 28.5, 23.5 / 22.6; twice 598 x 1019 x 3125, 250 tiles, 27.0 / 26.2, 24.1 / 20.4).
  // Onto bf16 results over up to five steps an element a lane, which odd rows leave, is the slower end (1749 x 173
  // x 1407 11.9 / 14.7, 11.2 / 12.2).
  // From a row-major B of rows that start on words the lines are touched once more by A alone: to 46 steps (1332 x
  // 1992 x 1783 36.5 / 33.8, 30.1 / 26.3, twice 429 x 2894 x 3511, 46 of them, 46.2 / 44.9, 43.9 / 35.2, 1768 x
  // 2696 x 1679 43.0 / 43.1, 34.6 / 32.3; past them 1222 x 3074 x 1065 twice 41.7 / 45.7, 40.0 / 37.3; odd rows of
  // A 2387 x 2641 x 1031 37.0 / 47.2, 34.8 / 35.1, 1366 x 2257 x 2332 33.4 / 37.0, 31.6 / 27.9).
  // Past a round of 128 x 128 the copies' tiles take two: from a row-major B up to 32 steps (2491 x 1862 x 2026
  // 41.1 / 38.5, 38.8 / 31.3, odd rows of A 2072 x 1899 x 2689 43.3 / 43.6, 41.8 / 37.7; rows on words gain up to
  // 46, 1084 x 2582 x 2596 twice 51.7 / 46.6, 49.7 / 39.6, 1001 x 2050 x 4425 41.1 / 40.9, 40.5 / 34.1, and stay
  // with the copies all the same, whose route tests/test_plan_routes.py holds fast for the last; odd ones lose
  // there, 2103 x 2583 x 2065 43.2 / 54.3, 42.1 / 44.2), a k-fastest B up to 20 (547 x 1118 x 4107 twice 36.8 /
  // 31.7, 33.9 / 27.1; 2138 x 1460 x 2320 30.7 / 33.3, 28.6 / 26.3), with odd rows 16 (2146 x 927 x 2260 31.1 /
  // 29.9, 28.3 / 23.5; 894 x 1195 x 2688 twice 31.6 / 33.9, 29.5 / 27.0); up to six steps they are even (2057 x 323
  // x 2231 17.9 / 19.5, 16.2 / 16.8).
  // Over 79 random sizes of these classes 1.20 times as fast with three sets, 1.06 from memory (geometric means;
  // least 1.00 and 0.90).  Of one and two entries, as measured.
  const uint64_t large = tiles(128, 128);
  const bool words = g.lda % 2 == 0 && (!g.b_kmajor || g.ldb % 2 == 0);
  // int8 rows on words, or on pairs of bytes up to 16 steps (from memory and with three sets): k-fastest B from five
  // steps to 34, 875 x 3964 x 2980 35.6 / 31.6, 35.0 / 25.9, 1688 x 524 x 1292 14.5 / 12.3, 13.5 / 10.3, pairs 945 x
  // 1058 x 3508 19.7 / 17.7, 18.9 / 15.1, 1247 x 1158 x 2125 19.7 / 20.3, 18.2 / 16.4; past those pairs 1329 x 4210 x
  // 1494 33.4 / 39.7, 32.2 / 31.0; four steps 697 x 504 x 2771 13.4 / 14.1, 12.0 / 11.8.  A row-major B past a round
  // of 128 x 128, of pairs too: 2225 x 1010 x 2684 26.4 / 23.7, 25.9 / 19.6, 2816 x 1812 x 1415 32.6 / 33.7, 31.7 /
  // 27.7, 1291 x 4236 x 3778 52.4 / 50.7, 51.3 / 42.4.  Below, rows on pairs are as fast either way (2040 x 866 x
  // 1246 15.2 / 17.3, 14.2 / 13.8); rows on words would gain (1857 x 2008 x 1725 26.9 / 26.4, 25.3 / 20.9) and stay
  // with the copies, whose route tests/test_plan_routes.py holds fast for 1500 x 1000 x 1500.  Over 24 random sizes
  // of these classes 1.10 times as fast from memory, 1.22 with three sets (geometric means; least 0.97 and 1.08).
  if (kind != 2) {
    const uint64_t either = uint64_t(g.lda) | (g.b_kmajor ? uint64_t(g.ldb) : 0);
    if (g.batch > 2 || steps < 5 || either % 2 != 0 || steps > (g.b_kmajor && either % 4 != 0 ? 16u : 34u)) return 0;
    if (large <= units) return g.b_kmajor && g.n >= 128 ? 128 : 0;
  } else if (large > units) {
    if (g.batch > 2 || steps <= 6 || steps > (g.b_kmajor ? (words ? 20u : 16u) : 32u)) return 0;
  }
  if (large > units) {
    return g.n >= 160 && tiles(128, 160) <= units ? 160 : g.n >= 192 && tiles(128, 192) <= units ? 192 : 0;
  }
  if (g.n < 128 || (g.accum && g.c_bf16 && steps <= 5 && (g.lda % 2 != 0 || g.ldb % 2 != 0))) return 0;
  return steps <= (odd_rows && 3 * large <= 2 * units ? 15u : words && !g.b_kmajor && g.batch <= 2 ? 46u : 24u) ? 128 : 0;
}

hipError_t launch_gemm_ring_rows(const GemmArgs &g, int kind, hipStream_t stream) {
  GemmArgs whole = g;
  if (g.k_total != 0) whole.batch = 1, whole.k = g.k_total;   // the tile goes by the whole problem
  const uint32_t bn = gemm_ring_rows_columns(whole, kind);
  switch (kind) {
    case 0: return launch_kind<I8, false>(g, bn, stream);
    case 1: return launch_kind<I8, true>(g, bn, stream);
    case 2: return launch_kind<BF16, false>(g, bn, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mrl
