// Move between layouts with neither a shared contiguous run nor two long contiguous dims: the tile kernel, for sources of SE bytes an
// element (move_gather_1.hip, _2, _4: its forms are many, and a translation unit for each compiles beside the others).
#pragma once
#include "move_device.h"
#include "plan.h"

namespace mrl {
namespace {

// Any other pair of contiguous digits (an OddEven digit on one side, a Packed digit of rows: too
// short for the 64 x 64 transpose): a tile of up to 4096 elements, chosen on the host so that it
// holds long runs on both sides, is read in source order, converted in registers, and written
// in destination order out of LDS.  VS, VD: elements per access on the two sides, 4 or 2 where the
// element's neighbours in the tile are its neighbours in memory, else 1.  The loads of a batch of
// four accesses are in flight together, and their digits are worked out once per access, not per
// element: that arithmetic is what bounds the kernel.  Runs of two: bf16 18 x 123556 transposed 8.0 us, element by element on
// that side 11.7; f32 [16, 2, 5, 84558] to [0, 3, 2, 1] 23.3, 37.2.  NACT: digits that the tile extends along at most, a
// form each up to five: f32 [1189, 5, 2, 4, 82] to [3, 4, 0, 2, 1, 3oe2], five of them, takes 26.1 us (16.4 with the runs of two) and 69.6 as any
// number; two or three digits in the form for four take 8 to 20 % longer (f32 246041 x 5 x 5 transposed within 21.6 us, 17.6).
template <int SE, int DE, int VS, int VD, int NACT>
__global__ __launch_bounds__(256) void k_move_gather(MoveTile p) {
  __shared__ uint32_t lds[MOVE_TILE_MAX + MOVE_TILE_MAX / 32];
  int64_t base_s, base_d;
  uint32_t room[MOVE_MAX_RANK];
  tile_origin(p, base_s, base_d, room);
  auto cell = [](uint32_t t) { return t + t / 32; };
  constexpr int BATCH = 4;
  for (uint32_t t0 = 0; t0 < p.tile; t0 += 256 * VS * BATCH) {
    uint32_t raw[BATCH][VS];
#pragma unroll
    for (int u = 0; u < BATCH; u++) {
      const uint32_t t = t0 + (u * 256 + threadIdx.x) * VS;
      uint32_t so = 0;
      bool inside = t < p.tile;
#pragma unroll
      for (int d = 0; d < NACT; d++) {
        const uint32_t q = div_small(t, p.tstride_s[d], p.inv_s[d]);
        const uint32_t c = q - div_small(q, p.ext[d], p.inv_ext[d]) * p.ext[d];
        inside = inside && c < room[d];
        so += c * uint32_t(p.ss[d]);
      }
      load_run<SE, VS>(p.src, base_s + (inside ? so : 0u), raw[u]);
    }
    with_dtypes<SE, DE>(p.sdt, p.ddt, [&](auto sd, auto dd) {
#pragma unroll
      for (int u = 0; u < BATCH; u++)
#pragma unroll
        for (int e = 0; e < VS; e++) raw[u][e] = convert_raw(raw[u][e], decltype(sd)::value, decltype(dd)::value);
    });
#pragma unroll
    for (int u = 0; u < BATCH; u++) {
      const uint32_t t = t0 + (u * 256 + threadIdx.x) * VS;
      if (t < p.tile) {
#pragma unroll
        for (int e = 0; e < VS; e++) lds[cell(t) + e] = raw[u][e];  // a run of four never crosses a multiple of 32
      }
    }
  }
  __syncthreads();
#pragma unroll 4
  for (uint32_t t = threadIdx.x * VD; t < p.tile; t += 256 * VD) {
    uint32_t d_o = 0, at = 0;
    bool inside = true;
#pragma unroll
    for (int d = 0; d < NACT; d++) {
      const uint32_t q = div_small(t, p.tstride_d[d], p.inv_d[d]);
      const uint32_t c = q - div_small(q, p.ext[d], p.inv_ext[d]) * p.ext[d];
      inside = inside && c < room[d];
      d_o += c * uint32_t(p.ds[d]);
      at += c * p.tstride_s[d];
    }
    uint32_t v[VD];
#pragma unroll
    for (int e = 0; e < VD; e++) v[e] = lds[cell(at + (VD == 1 ? 0 : p.lds_step[e]))];
    if (inside) store_run<DE, VD>(p.dst, base_d + d_o, v);
  }
}
template <int SE, int DE, int VS, int VD>
hipError_t launch_runs(const MoveTile &t, uint32_t n_act, dim3 grid, hipStream_t stream) {
  if (n_act <= 2) MRL_LAUNCH((k_move_gather<SE, DE, VS, VD, 2>), grid, dim3(256), 0, stream, t);
  else if (n_act <= 3) MRL_LAUNCH((k_move_gather<SE, DE, VS, VD, 3>), grid, dim3(256), 0, stream, t);
  else if (n_act <= 4) MRL_LAUNCH((k_move_gather<SE, DE, VS, VD, 4>), grid, dim3(256), 0, stream, t);
  else if (n_act <= 5) MRL_LAUNCH((k_move_gather<SE, DE, VS, VD, 5>), grid, dim3(256), 0, stream, t);
  else MRL_LAUNCH((k_move_gather<SE, DE, VS, VD, int(MOVE_MAX_RANK)>), grid, dim3(256), 0, stream, t);
  return plan::last_error();
}
// (two elements of a byte go one by one: two bytes are no wider an access than one)
template <int SE, int DE, int VS>
hipError_t launch_from(const MoveTile &t, uint32_t run_d, uint32_t n_act, dim3 grid, hipStream_t stream) {
  if (run_d == 4) return launch_runs<SE, DE, VS, 4>(t, n_act, grid, stream);
  if (run_d == 2) return launch_runs<SE, DE, VS, (DE > 1 ? 2 : 1)>(t, n_act, grid, stream);
  return launch_runs<SE, DE, VS, 1>(t, n_act, grid, stream);
}
template <int SE, int DE>
hipError_t launch_to(const MoveTile &t, uint32_t run_s, uint32_t run_d, uint32_t n_act, dim3 grid, hipStream_t stream) {
  if (run_s == 4) return launch_from<SE, DE, 4>(t, run_d, n_act, grid, stream);
  if (run_s == 2) return launch_from<SE, DE, (SE > 1 ? 2 : 1)>(t, run_d, n_act, grid, stream);
  return launch_from<SE, DE, 1>(t, run_d, n_act, grid, stream);
}
}  // namespace

template <int SE>
hipError_t launch_move_gather(const MoveTile &t, uint32_t dst_bytes, uint32_t run_s, uint32_t run_d, uint32_t n_act, uint32_t blocks, hipStream_t stream) {
  if (dst_bytes == 1) return launch_to<SE, 1>(t, run_s, run_d, n_act, dim3(blocks), stream);
  if (dst_bytes == 2) return launch_to<SE, 2>(t, run_s, run_d, n_act, dim3(blocks), stream);
  return launch_to<SE, 4>(t, run_s, run_d, n_act, dim3(blocks), stream);
}

}  // namespace mrl
