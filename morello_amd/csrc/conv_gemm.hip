// Conv as an implicit Matmul on the matrix cores: the kernels of gemm_mfma_kernel.h and of
// gemm_ring_tile.h with their left operand addressed as the windows of a channels-last image (the CONV build) and the KRSC
// filters as a B operand stored k-fastest.  Takes any Conv whose channel vectors are whole
// 16-byte chunks (morello/src/spec.rs:486-494: no stride, no padding); nothing is unfolded in
// memory.  Its own translation unit so that the instantiations compile beside the others.
#include "gemm_mfma_kernel.h"
#include "gemm_ring_tile.h"

namespace mrl {
namespace {
using namespace gemm;

typedef Tile<64, 64, 128, 2, 2> T64;

template <class T, bool A_UNSIGNED>
hipError_t launch_for(const GemmArgs &g, uint32_t tile, hipStream_t stream) {
  if (tile == 64) return launch<T, A_UNSIGNED, T64, true, true, true>(g, stream);
  if (tile == 128) return launch<T, A_UNSIGNED, Tile128<T, true>, true, true, true>(g, stream);
  return launch<T, A_UNSIGNED, TileBig, true, true, true>(g, stream);
}

// The tiles of gemm_ring_tile.h on windows: 32 RA pixels by 32 RB filters on eight waves, two to a SIMD, each with
// half of every step.
template <class T, bool A_UNSIGNED, int RA, int RB, bool CONV, int SLOTS>
__global__ __launch_bounds__(64 * ring::WAVES, RA * RB <= 8 ? 4 : 2) void k_gemm(MRL_WALK_PARAMS, GemmArgs g) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  MRL_WALK_TILE(tile_m, tile_n)
  ring::ring_tile<T, A_UNSIGNED, true, RA, RB, SLOTS, CONV>(lds, tile_m, tile_n, g);
}
template <class T, bool A_UNSIGNED, int RA, int RB, bool CONV, int SLOTS>
hipError_t launch_ring_tile(const GemmArgs &g, hipStream_t stream) {
  constexpr int BM = 32 * RA, BN = 32 * RB, LDS = SLOTS * (BM + BN) * ring::STEP;
  static_assert(LDS >= 4 * 16 * RA * (16 * RB + 4) * 4, "the waves' pieces of C fit");
  static std::atomic<uint64_t> lds_limit_set{0};
  if (!plan::recording() && LDS > 65536) {
    hipError_t e = raise_lds_limit(lds_limit_set, (const void *)k_gemm<T, A_UNSIGNED, RA, RB, CONV, SLOTS>, LDS);
    if (e != hipSuccess) return e;
  }
  const int tiles_m = int((g.m + BM - 1) / BM), tiles_n = int((g.n + BN - 1) / BN);
  const double mn = double(g.m) * g.n * g.batch, steps = double((uint64_t(g.k) * T::ES + ring::STEP - 1) / ring::STEP);
  plan::work(T::ES == 1 ? plan::UNIT_MFMA_I8 : plan::UNIT_MFMA_BF16, 2.0 * mn * g.k,
             double(g.conv.image_bytes) + double(g.n) * (g.k_total ? g.k_total : g.k) * T::ES + mn * 4 * (g.accum ? 2 : 1),
             2.0 * BM * BN * steps * (ring::STEP / T::ES), RA * RB > 4 ? 2500.0 + 300.0 * steps : 1300.0 + (T::ES == 2 ? 145.0 : 210.0) * steps);
  const TileWalk walk = gemm::tile_walk(tiles_m, tiles_n);
  MRL_LAUNCH((k_gemm<T, A_UNSIGNED, RA, RB, CONV, SLOTS>), dim3(tiles_m * tiles_n, g.batch), dim3(64 * ring::WAVES), LDS, stream, MRL_WALK_ARGS(walk), g);
  return plan::last_error();
}

// Where those tiles are the faster ones.  A launch's time is taken as a fixed part and, for every round of its
// workgroups over the compute units, the steps of a workgroup (128 bytes of the windows).  Measured (us; a step and
// round, int8 / bf16):
//   these tiles: 64 x 32 3.5 + 0.25 / 0.24 (a single round 0.18 / 0.13), 64 x 64 3.5 + 0.26 / 0.25 (0.22 / 0.15), 128
//     x 32 4 + 0.30 / 0.29, 128 x 64 4.5 + 0.31 / 0.32 (a single round of bf16 0.25), 128 x 128 5.5 + 0.48 / 0.50,
//     128 x 192 6.5 + 0.66 / 0.67; int8 past one round of the last two 0.66 and 0.89, to one and a half of 128 x 64
//     0.43, and the same beside the 256 x 256 tile: nothing is under way while a round's results leave, which a short
//     int8 step does not make up for (u8 18 x (208 -> 240) x 71^2 3 x 3 74.5 / 91.3, 18 x (176 -> 192) x 79^2 65.1 /
//     73.1, 22 x (208 -> 64) x 46^2 15.6 / 17.7, 16 x (112 -> 160) x 55^2 20.8 / 25.1),
//   k_gemm's: 64 3.5 + 0.30 / 0.245, 128 4 + 0.69 / 0.57, 256 5 + 2.15 / 1.83;
// past the third round those of which several share a unit even out the last one.  What bounds a single round is the
// wait for what the step after next asked of memory, past one the way into LDS.  (us, k_gemm / this: bf16 12 x (352
// -> 192) x 68^2 5 x 5 265.7 / 190.5, u8 18 x (272 -> 192) x 42^2 5 x 5 101.9 / 55.2, 9 x (224 -> 304) x 27^2 5 x 5
// 33.0 / 27.1, 5 x (144 -> 112) x 64^2 5 x 5 23.1 / 19.4, bf16 11 x (144 -> 208) x 14^2 3 x 3 10.3 / 7.5.  Windows by
// way of registers, two slots of LDS / straight to LDS, three or four: bf16 21 x (144 -> 64) x 17^2 3 x 3 7.5 / 6.4,
// 2 x (96 -> 48) x 69^2 6.3 / 5.6, u8 31 x (240 -> 144) x 14^2 5 x 5 23.2 / 19.6, 1 x (64 -> 48) x 21^2 5 x 5 6.1 /
// 5.7; over 140 random layers 1.035 times as fast.)
// Few steps leave the start and the end of a workgroup, and k_gemm's are the shorter ones (us, k_gemm / 64 x 64 or
// 128 x 64 of these, whichever is the faster): one step, whatever the number of tiles, u8 4 x (32 -> 128) x 28^2 2 x
// 2 3.3 / 3.9, bf16 8 x (8 -> 128) x 40^2 2 x 2 3.6 / 5.2; up to three in one round, where it is even at the last (u8
// 2 x (32 -> 64) x 28^2 3 x 3 4.0 / 4.1), u8 4 x (16 -> 176) x 57^2 3 x 3, two, 6.0 / 7.7; up to seven past one, 28 x
// (48 -> 336) x 11^2, four, 5.8 / 6.1, bf16 30 x (32 -> 96) x 18^2, five, 5.1 / 5.5, 20 x (16 -> 128) x 28^2, three,
// 4.7 / 5.9.  But for its 256 x 256 tile, whose end is the longer one: u8 7 x (16 -> 272) x 72^2 3 x 3, two steps,
// 27.6 / 19.1, bf16 17 x (16 -> 176) x 70^2 5 x 5, seven, 36.6 / 28.7.
// Of int8 where that tile pads the filters half as much again (without, 22 x (16 -> 176) x 114^2 3 x 3 61.4 / 84.4,
// 22 x (48 -> 208) x 40^2 15.3 / 19.1), and not for two steps past fourteen rounds, which the results bound (27 x (16
// -> 288) x 71^2 53.0 / 60.9).
enum Tiles : uint32_t { SQUARE, T64x32, T64x64, T128x32, T128x64, T128x128, T128x192 };
Tiles choose_tiles(const GemmArgs &g, int kind) {
  if (kind > 2) return SQUARE;
  const uint64_t es = kind == 2 ? 2 : 1, step = ring::STEP, steps = (uint64_t(g.k) * es + step - 1) / step;
  const uint64_t last = g.k_total != 0 ? g.k_total - uint64_t(g.batch - 1) * g.k : g.k;
  if (last * es <= step) return SQUARE;
  const uint64_t units = g_compute_units;
  auto tiles = [&](uint32_t bm, uint32_t bn) { return uint64_t((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * g.batch; };
  const uint64_t small = tiles(64, 64);
  if (small <= units) {
    if (steps < 4 && g.batch == 1) return SQUARE;
    // (two columns of 32 for up to 48 filters where the chip has room for both: u8 3 x (272 -> 48) x 8^2 5 x 5 8.7 / 7.7)
    return g.n <= 32 || (g.n <= 48 && 2 * small <= units) ? T64x32 : T64x64;
  }
  const uint32_t side = gemm_tile_side(g, kind);
  if (g.batch > 1 || (steps < 8 && side != 256)) return SQUARE;   // (slices three to a unit: bf16 26 x (336 -> 80) x 11^2 in six 13.5 / 14.4)
  const bool i8 = kind != 2;
  if (i8 && steps < 8 && (16 * tiles(256, 256) <= 3 * tiles(128, 64) || (steps == 2 && tiles(128, 64) > 14 * units))) return SQUARE;
  auto us = [&](uint32_t bm, uint32_t bn, bool shared, double fixed, double step_us) {
    const double r = double(tiles(bm, bn)) / double(units), whole = double((tiles(bm, bn) + units - 1) / units);
    return fixed + double(steps) * step_us * (shared && r > 3.0 ? (r + whole) / 2 : whole);
  };
  Tiles best = SQUARE;
  double least = 1e300;
  auto consider = [&](Tiles t, double time) {
    if (time < least) best = t, least = time;
  };
  if (g.n <= 32) {
    consider(T128x32, us(128, 32, true, 4.0, i8 ? 0.30 : 0.29));
    consider(T64x32, us(64, 32, true, 3.5, (i8 ? 0.25 : 0.24) * (tiles(64, 32) > 3 * units ? 0.8 : 1.0)));
  } else {
    if (g.n <= 64) consider(T64x64, us(64, 64, true, 3.5, i8 ? 0.26 : 0.25));
    const uint64_t t = tiles(128, 64);
    const bool slow = (side == 256 && steps >= 8) || (t > units && 2 * t <= 3 * units);   // (int8)
    consider(T128x64, us(128, 64, true, 4.5, (i8 ? (slow ? 0.43 : 0.31) : t > units ? 0.32 : 0.25) * (t > 2 * units ? 1.08 : 1.0)));
    if (g.n > 64 && steps >= 12) {
      consider(T128x128, us(128, 128, false, 5.5, !i8 ? 0.50 : tiles(128, 128) > units ? 0.66 : 0.48));
      consider(T128x192, us(128, 192, false, 6.5, !i8 ? 0.67 : tiles(128, 192) > units ? 0.89 : 0.66));
    }
  }
  const double square = side == 64    ? us(64, 64, true, 3.5, i8 ? 0.30 : 0.245)
                        : side == 128 ? us(128, 128, true, 4.0, (i8 ? 0.69 : 0.57) * (tiles(128, 128) > units ? 0.87 : 1.0))
                                      : us(256, 256, false, 5.0, i8 ? 2.15 : 1.83);
  return least < 0.85 * square ? best : SQUARE;   // (the times above are within a seventh of what a layer takes)
}

template <class T, bool A_UNSIGNED>
hipError_t launch_tiles(const GemmArgs &g, Tiles tiles, hipStream_t stream) {
  switch (tiles) {
    case T64x32: return launch_ring_tile<T, A_UNSIGNED, 2, 1, true, 4>(g, stream);
    case T64x64: return launch_ring_tile<T, A_UNSIGNED, 2, 2, true, 4>(g, stream);
    case T128x32: return launch_ring_tile<T, A_UNSIGNED, 4, 1, true, 4>(g, stream);
    case T128x64: return launch_ring_tile<T, A_UNSIGNED, 4, 2, true, 3>(g, stream);
    case T128x128: return launch_ring_tile<T, A_UNSIGNED, 4, 4, true, 4>(g, stream);
    default: return launch_ring_tile<T, A_UNSIGNED, 4, 6, true, 4>(g, stream);
  }
}

}  // namespace

bool conv_gemm_applicable(const GemmArgs &g, int kind) {
  const int es = kind == 3 ? 4 : kind == 2 ? 2 : 1;
  auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  return g.b_kmajor && (g.batch == 1 || (g.conv.slice_bytes != 0 && g.conv.slice_bytes % 16 == 0)) && g.conv.c_bytes != 0 && g.conv.c_bytes % 16 == 0 &&
         g.conv.image_bytes < (1ull << 31) && g.m >= 1 && g.n >= 1 && g.k >= 1 && g.ldb % (16 / es) == 0 &&
         al16(g.a) && al16(g.b) && (reinterpret_cast<uintptr_t>(g.c) & 3) == 0 && edge_addressable(g, es) &&
         uint64_t((g.m + 63) / 64) * ((g.n + 63) / 64) < (1u << 30);
}

hipError_t launch_conv_gemm(const GemmArgs &args, int kind, hipStream_t stream, uint32_t tile) {
  if (!conv_gemm_applicable(args, kind) || (tile != 0 && tile != 64 && tile != 128 && tile != 256)) return hipErrorInvalidValue;
  // Pixel numbers and window bytes stay below 2^31 (conv_gemm_applicable), as FastDiv asks.
  GemmArgs g = args;
  g.conv.by_ow = FastDiv(g.conv.ow), g.conv.by_oh = FastDiv(g.conv.oh);
  g.conv.by_c_bytes = FastDiv(g.conv.c_bytes), g.conv.by_fw = FastDiv(g.conv.fw);
  g.conv.by_run = FastDiv(g.conv.fw * g.conv.c_bytes), g.conv.run_gap = (g.conv.w - g.conv.fw) * g.conv.c_bytes;
  if (tile == 0) {
    if (const Tiles tiles = choose_tiles(g, kind); tiles != SQUARE) {
      switch (kind) {
        case 0: return launch_tiles<I8, false>(g, tiles, stream);
        case 1: return launch_tiles<I8, true>(g, tiles, stream);
        default: return launch_tiles<BF16, false>(g, tiles, stream);
      }
    }
    tile = g.conv.slice_bytes != 0 ? 64 : gemm_tile_side(g, kind);
  }
  switch (kind) {
    case 0: return launch_for<I8, false>(g, tile, stream);
    case 1: return launch_for<I8, true>(g, tile, stream);
    case 2: return launch_for<BF16, false>(g, tile, stream);
    case 3: return launch_for<F32, false>(g, tile, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mrl
