// Correctness-first kernels: any dtype combination, any strides, any size.  The MFMA
// kernels cover the shapes that matter for throughput; everything else lands here so that
// every Spec the descriptor can express still runs on the GPU.
//
// Arithmetic follows the reference's oracle (morello/src/verification.rs:115-134,
// 547-569, 603-643): both inputs are converted to the output dtype, then multiplied and
// accumulated in that dtype.  Integer outputs are computed modulo 2^32 and truncated on
// store, which equals wrapping arithmetic in the narrower type.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "kernels.h"
#include "layout_factor.h"
#include "move_device.h"
#include "pad_position.h"
#include "row_chunks.h"

namespace mrl {
namespace {

__device__ inline float load_f32(const void *p, int dtype, int64_t off) {
  switch (dtype) {
    case MRL_U8: return float(((const uint8_t *)p)[off]);
    case MRL_I8: return float(((const int8_t *)p)[off]);
    case MRL_U16: return float(((const uint16_t *)p)[off]);
    case MRL_I16: return float(((const int16_t *)p)[off]);
    case MRL_U32: return float(((const uint32_t *)p)[off]);
    case MRL_I32: return float(((const int32_t *)p)[off]);
    case MRL_F32: return ((const float *)p)[off];
    default: return bf16_bits_to_f32(((const uint16_t *)p)[off]);
  }
}

// Rust `as` semantics (verification.rs:547-569, `x.as_()` into the output dtype): integers wrap,
// floats saturate at the bounds of the dtype they are cast to and NaN becomes 0.
__device__ inline uint32_t load_u32(const void *p, int dtype, int64_t off, int out_dtype) {
  uint32_t v;
  switch (dtype) {
    case MRL_U8: v = ((const uint8_t *)p)[off]; break;
    case MRL_I8: v = uint32_t(int32_t(((const int8_t *)p)[off])); break;
    case MRL_U16: v = ((const uint16_t *)p)[off]; break;
    case MRL_I16: v = uint32_t(int32_t(((const int16_t *)p)[off])); break;
    case MRL_U32: v = ((const uint32_t *)p)[off]; break;
    case MRL_I32: v = uint32_t(((const int32_t *)p)[off]); break;
    default: v = float_to_int(load_f32(p, dtype, off), out_dtype);
  }
  return narrow_int(out_dtype, v);
}

__device__ inline void store_u32(void *p, int dtype, int64_t off, uint32_t v) {
  switch (dtype) {
    case MRL_U8: case MRL_I8: ((uint8_t *)p)[off] = uint8_t(v); break;
    case MRL_U16: case MRL_I16: case MRL_BF16: ((uint16_t *)p)[off] = uint16_t(v); break;
    default: ((uint32_t *)p)[off] = v; break;
  }
}

// ------------------------------------------------------------------ relayout
__global__ void k_relayout(const uint8_t *src, uint8_t *dst, LayoutEval sl, LayoutEval dl,
                           uint32_t es, uint64_t count) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint32_t pt[MRL_MAX_RANK];
  uint64_t rem = i;
  for (int d = int(sl.rank) - 1; d >= 0; d--) {
    pt[d] = uint32_t(rem % sl.shape[d]);
    rem /= sl.shape[d];
  }
  const int64_t so = layout_offset(sl, pt), d_o = layout_offset(dl, pt);
  if (es == 1) dst[d_o] = src[so];
  else if (es == 2) ((uint16_t *)dst)[d_o] = ((const uint16_t *)src)[so];
  else ((uint32_t *)dst)[d_o] = ((const uint32_t *)src)[so];
}

// ---------------------------------------------------------------------- move
// One element: read as `sdt`, converted with Rust `as` semantics, returned as the bits of `ddt`.
__device__ inline uint32_t move_bits(const void *src, int sdt, int64_t so, int ddt) {
  if (sdt == ddt) {  // bits as they are (a NaN keeps its payload)
    const size_t size = sdt == MRL_U8 || sdt == MRL_I8 ? 1 : sdt == MRL_U16 || sdt == MRL_I16 || sdt == MRL_BF16 ? 2 : 4;
    return size == 1 ? ((const uint8_t *)src)[so] : size == 2 ? ((const uint16_t *)src)[so] : ((const uint32_t *)src)[so];
  }
  const bool src_float = sdt == MRL_F32 || sdt == MRL_BF16;
  if (ddt == MRL_F32) return __float_as_uint(load_f32(src, sdt, so));
  if (ddt == MRL_BF16) return f32_to_bf16_bits(load_f32(src, sdt, so));
  if (src_float) return float_to_int(load_f32(src, sdt, so), ddt);
  return load_u32(src, sdt, so, MRL_U32);  // int -> int wraps
}

// Move of a contiguous run with a dtype conversion: N elements per thread, one vector load
// and one vector store (SE, DE: element sizes in bytes).  N = 4 where an element of four bytes is
// involved, 8 or 16 between narrower ones, so that the wider side moves 16 bytes a thread (u8 ->
// bf16 over 64 Mi elements: 68 us with four elements a thread).
template <int SE, int DE, int N = 4>
__global__ __launch_bounds__(256) void k_convert4(const void *__restrict__ src, void *__restrict__ dst, int sdt,
                                                  int ddt, uint64_t count) {
  // A pack travels as whole dwords (loads and stores of 4, 8 or 16 bytes, two of 16 for a pack of
  // 32), and an element is cut out of its dword by shifts: through arrays of bytes the compiler
  // narrowed the load of a u16 -> u8 pack to the sixteen bytes the conversion keeps, one load each.
  constexpr int SW = SE * N / 4, DW = DE * N / 4;   // dwords of a pack on either side
  static_assert(SE * N % 4 == 0 && DE * N % 4 == 0, "packs are whole dwords");
  struct alignas(SW >= 4 ? 16 : SW * 4) SrcPack { uint32_t w[SW]; };
  struct alignas(DW >= 4 ? 16 : DW * 4) DstPack { uint32_t w[DW]; };
  const uint64_t packs = count / N, step = uint64_t(gridDim.x) * 256;
  // (the dtypes are switched on once per pack: with_dtypes)
  auto convert_pack = [&](const SrcPack &in, DstPack &out, auto sd, auto dd) {
#pragma unroll
    for (int w = 0; w < DW; w++) out.w[w] = 0;
#pragma unroll
    for (int e = 0; e < N; e++) {
      const uint32_t raw = SE == 4 ? in.w[e] : (in.w[e * SE / 4] >> (8 * (e * SE % 4))) & (SE == 1 ? 0xffu : 0xffffu);
      const uint32_t v = convert_raw(raw, decltype(sd)::value, decltype(dd)::value);
      if constexpr (DE == 4) out.w[e] = v;
      else out.w[e * DE / 4] |= (v & (DE == 1 ? 0xffu : 0xffffu)) << (8 * (e * DE % 4));
    }
  };
  for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < packs; i += step) {
    SrcPack in;
    if constexpr (SW == 1) in.w[0] = static_cast<const uint32_t *>(src)[i];
    else if constexpr (SW == 2) { const v2u v = static_cast<const v2u *>(src)[i]; in.w[0] = v[0], in.w[1] = v[1]; }
    else {
#pragma unroll
      for (int q = 0; q < SW / 4; q++) {
        const v4u_t v = static_cast<const v4u_t *>(src)[i * (SW / 4) + q];
#pragma unroll
        for (int k = 0; k < 4; k++) in.w[q * 4 + k] = v[k];
      }
    }
    DstPack out;
    with_dtypes<SE, DE>(sdt, ddt, [&](auto sd, auto dd) { convert_pack(in, out, sd, dd); });
    // the converted elements as one store of 4, 8 or 16 bytes
    static_assert(DW == 1 || DW == 2 || DW == 4, "a pack is stored by one instruction");
    if constexpr (DW == 1) MRL_STORE_ONCE(out.w[0], static_cast<uint32_t *>(dst) + i);
    else if constexpr (DW == 2) MRL_STORE_ONCE((v2u{out.w[0], out.w[1]}), static_cast<v2u *>(dst) + i);
    else MRL_STORE_ONCE((v4u_t{out.w[0], out.w[1], out.w[2], out.w[3]}), static_cast<v4u_t *>(dst) + i);
  }
  // The elements past the last whole pack.
  if (blockIdx.x == 0 && threadIdx.x < count % N) {
    const int64_t at = int64_t(packs * N + threadIdx.x);
    store_u32(dst, ddt, at, move_bits(src, sdt, at, ddt));
  }
}

__global__ void k_move_generic(const void *src, void *dst, LayoutEval sl, LayoutEval dl, int sdt,
                               int ddt, uint64_t count) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint32_t pt[MRL_MAX_RANK];
  uint64_t rem = i;
  for (int d = int(sl.rank) - 1; d >= 0; d--) {
    pt[d] = uint32_t(rem % sl.shape[d]);
    rem /= sl.shape[d];
  }
  const int64_t so = layout_offset(sl, pt), d_o = layout_offset(dl, pt);
  store_u32(dst, ddt, d_o, move_bits(src, sdt, so, ddt));
}

// Move between two layouts that are permutations of the logical dims (element strides on both
// sides).  `order` lists the dims slowest to fastest for the index decode.
struct MoveStrided {
  const void *src;
  void *dst;
  int sdt, ddt;
  uint32_t rank;
  uint32_t shape[MOVE_MAX_RANK];
  int64_t ss[MOVE_MAX_RANK], ds[MOVE_MAX_RANK];
  uint32_t order[MOVE_MAX_RANK];
  uint32_t dim_s, dim_d;      // the dim each side stores contiguously
  uint32_t tiles_s, tiles_d;  // 64-element tiles along them
  uint64_t count;
  FastDiv by_shape[MOVE_MAX_RANK];   // by shape[order[o]], for place_of (a tensor has fewer than 2^31 elements)
};

// Where the i-th element (or vector) in destination order lies on the two sides.
__device__ inline void place_of(const MoveStrided &p, uint32_t i, int64_t &so, int64_t &d_o) {
  so = d_o = 0;
  for (int o = int(p.rank) - 1; o >= 0; o--) {
    const uint32_t d = p.order[o], rest = p.by_shape[o].div(i), c = i - rest * p.shape[d];
    i = rest;
    so += int64_t(c) * p.ss[d], d_o += int64_t(c) * p.ds[d];
  }
}

// Both sides contiguous along the same dim: consecutive threads take consecutive elements of
// that dim, so reads and writes are both coalesced.
__global__ __launch_bounds__(256) void k_move_rows(MoveStrided p) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= p.count) return;
  int64_t so, d_o;
  place_of(p, uint32_t(i), so, d_o);  // (a tensor has fewer than 2^31 elements)
  store_u32(p.dst, p.ddt, d_o, move_bits(p.src, p.sdt, so, p.ddt));
}

// The two sides are contiguous along different dims: a 64 x 64 tile of (dim_d, dim_s) goes
// through LDS, read with dim_s fastest and written with dim_d fastest, so both sides see
// whole contiguous runs (move_relayout of morello/src/scheduling/moves.rs as a transpose).
template <int SE, int DE>
__global__ __launch_bounds__(256) void k_move_tiled(MoveStrided p) {
  __shared__ uint32_t tile[64][65];
  uint64_t blk = blockIdx.x;
  const uint32_t ts = uint32_t(blk % p.tiles_s);
  blk /= p.tiles_s;
  // Diagonal order: workgroups that run together differ in both tile coordinates.  In row or
  // column order they would all read (or all write) addresses a whole number of rows apart,
  // which with power-of-two row lengths is one memory channel for all of them.
  const uint32_t td = uint32_t((blk + ts) % p.tiles_d);
  blk /= p.tiles_d;
  // The remaining dims, slowest to fastest in `order` (dim_s and dim_d are skipped).
  int64_t so = 0, d_o = 0;
  for (int o = int(p.rank) - 1; o >= 0; o--) {
    const uint32_t d = p.order[o];
    if (d == p.dim_s || d == p.dim_d) continue;
    const uint32_t c = uint32_t(blk % p.shape[d]);
    blk /= p.shape[d];
    so += int64_t(c) * p.ss[d], d_o += int64_t(c) * p.ds[d];
  }
  const uint32_t lane = threadIdx.x & 63, quad = threadIdx.x >> 6;
  const uint32_t s0 = ts * 64, d0 = td * 64, ns = p.shape[p.dim_s], nd = p.shape[p.dim_d];
  // All sixteen loads of a thread are issued before the first is used: a small tensor is a
  // handful of tiles, and their time is these loads' latency.
  uint32_t v[16];
#pragma unroll
  for (uint32_t i = 0; i < 16; i++) {
    const uint32_t r = quad + 4 * i;
    v[i] = 0;
    if (d0 + r < nd && s0 + lane < ns)
      v[i] = load_sized<SE>(p.src, so + int64_t(d0 + r) * p.ss[p.dim_d] + int64_t(s0 + lane) * p.ss[p.dim_s]);
  }
  // The conversion is arithmetic on registers, after the loads: a dtype switch around each load
  // would put a branch between any two of them.
  with_dtypes<SE, DE>(p.sdt, p.ddt, [&](auto sd, auto dd) {
#pragma unroll
    for (uint32_t i = 0; i < 16; i++) tile[quad + 4 * i][lane] = convert_raw(v[i], decltype(sd)::value, decltype(dd)::value);
  });
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < 16; i++) {
    const uint32_t r = quad + 4 * i;
    if (s0 + r < ns && d0 + lane < nd)
      store_sized<DE>(p.dst, d_o + int64_t(s0 + r) * p.ds[p.dim_s] + int64_t(d0 + lane) * p.ds[p.dim_d], tile[lane][r]);
  }
}

// The same with nothing converted: typed loads and stores (the dtype switch of the converting
// form puts a branch between any two loads, so none of them overlap).
template <class E>
__global__ __launch_bounds__(256) void k_move_tiled_as(MoveStrided p) {
  __shared__ uint32_t tile[64][65];
  const E *src = static_cast<const E *>(p.src);
  E *dst = static_cast<E *>(p.dst);
  uint64_t blk = blockIdx.x;
  const uint32_t ts = uint32_t(blk % p.tiles_s);
  blk /= p.tiles_s;
  const uint32_t td = uint32_t((blk + ts) % p.tiles_d);
  blk /= p.tiles_d;
  // The remaining dims, slowest to fastest in `order` (dim_s and dim_d are skipped).
  int64_t so = 0, d_o = 0;
  for (int o = int(p.rank) - 1; o >= 0; o--) {
    const uint32_t d = p.order[o];
    if (d == p.dim_s || d == p.dim_d) continue;
    const uint32_t c = uint32_t(blk % p.shape[d]);
    blk /= p.shape[d];
    so += int64_t(c) * p.ss[d], d_o += int64_t(c) * p.ds[d];
  }
  const uint32_t lane = threadIdx.x & 63, quad = threadIdx.x >> 6;
  const uint32_t s0 = ts * 64, d0 = td * 64, ns = p.shape[p.dim_s], nd = p.shape[p.dim_d];
  uint32_t v[16];
#pragma unroll
  for (uint32_t i = 0; i < 16; i++) {
    const uint32_t r = quad + 4 * i;
    v[i] = 0;
    if (d0 + r < nd && s0 + lane < ns)
      v[i] = src[so + int64_t(d0 + r) * p.ss[p.dim_d] + int64_t(s0 + lane) * p.ss[p.dim_s]];
  }
#pragma unroll
  for (uint32_t i = 0; i < 16; i++) tile[quad + 4 * i][lane] = v[i];
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < 16; i++) {
    const uint32_t r = quad + 4 * i;
    if (s0 + r < ns && d0 + lane < nd)
      dst[d_o + int64_t(s0 + r) * p.ds[p.dim_s] + int64_t(d0 + lane) * p.ds[p.dim_d]] = E(tile[lane][r]);
  }
}

// The same transpose for 16-bit elements that are not converted: 128 x 128 tiles, two elements
// (one dword) per lane on both sides.  Needs even extents along both contiguous dims and even
// strides elsewhere, so that every dword is whole and aligned.
__global__ __launch_bounds__(256) void k_move_tiled16(MoveStrided p) {
  __shared__ uint16_t tile[128][130];
  uint64_t blk = blockIdx.x;
  const uint32_t ts = uint32_t(blk % p.tiles_s);
  blk /= p.tiles_s;
  const uint32_t td = uint32_t((blk + ts) % p.tiles_d);  // diagonal order, see k_move_tiled
  blk /= p.tiles_d;
  int64_t so = 0, d_o = 0;
  for (int o = int(p.rank) - 1; o >= 0; o--) {
    const uint32_t d = p.order[o];
    if (d == p.dim_s || d == p.dim_d) continue;
    const uint32_t c = uint32_t(blk % p.shape[d]);
    blk /= p.shape[d];
    so += int64_t(c) * p.ss[d], d_o += int64_t(c) * p.ds[d];
  }
  const uint32_t lane = threadIdx.x & 63, quad = threadIdx.x >> 6;
  const uint32_t s0 = ts * 128, d0 = td * 128, ns = p.shape[p.dim_s], nd = p.shape[p.dim_d];
  const uint16_t *src = static_cast<const uint16_t *>(p.src);
  uint16_t *dst = static_cast<uint16_t *>(p.dst);
#pragma unroll 4
  for (uint32_t r = quad; r < 128; r += 4)
    if (d0 + r < nd && s0 + 2 * lane < ns) {
      const uint32_t pair = *(const uint32_t *)(src + so + int64_t(d0 + r) * p.ss[p.dim_d] + (s0 + 2 * lane));
      tile[r][2 * lane] = uint16_t(pair), tile[r][2 * lane + 1] = uint16_t(pair >> 16);
    }
  __syncthreads();
#pragma unroll 4
  for (uint32_t r = quad; r < 128; r += 4)
    if (s0 + r < ns && d0 + 2 * lane < nd) {
      const uint32_t pair = uint32_t(tile[2 * lane][r]) | (uint32_t(tile[2 * lane + 1][r]) << 16);
      *(uint32_t *)(dst + d_o + int64_t(s0 + r) * p.ds[p.dim_s] + (d0 + 2 * lane)) = pair;
    }
}

// 16-bit elements whose source rows are whole 16-byte vectors: the 128 x 128 tile sits in LDS as
// dwords (pairs along the source's contiguous dim), loaded eight elements per lane; a lane then
// takes the dwords of two neighbouring tile rows and regroups their halves into the two dwords
// it stores (pairs along the destination's contiguous dim).  No 16-bit LDS access, no bank
// conflict beyond the two passes 64 lanes need anyway.
__global__ __launch_bounds__(256) void k_move_tiled16v(MoveStrided p) {
  __shared__ uint32_t tile[128][65];
  uint64_t blk = blockIdx.x;
  const uint32_t ts = uint32_t(blk % p.tiles_s);
  blk /= p.tiles_s;
  const uint32_t td = uint32_t((blk + ts) % p.tiles_d);  // diagonal order, see k_move_tiled
  blk /= p.tiles_d;
  int64_t so = 0, d_o = 0;
  for (int o = int(p.rank) - 1; o >= 0; o--) {
    const uint32_t d = p.order[o];
    if (d == p.dim_s || d == p.dim_d) continue;
    const uint32_t c = uint32_t(blk % p.shape[d]);
    blk /= p.shape[d];
    so += int64_t(c) * p.ss[d], d_o += int64_t(c) * p.ds[d];
  }
  typedef uint32_t quad_t __attribute__((ext_vector_type(4)));
  const uint32_t s0 = ts * 128, d0 = td * 128, ns = p.shape[p.dim_s], nd = p.shape[p.dim_d];
  const uint16_t *src = static_cast<const uint16_t *>(p.src);
  uint16_t *dst = static_cast<uint16_t *>(p.dst);
  const uint32_t col = (threadIdx.x & 15) * 8, row = threadIdx.x >> 4;
  quad_t v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const uint32_t r = row + 16 * i;
    v[i] = quad_t{0, 0, 0, 0};
    if (d0 + r < nd && s0 + col < ns)
      v[i] = MRL_LOAD_ONCE((const quad_t *)(src + so + int64_t(d0 + r) * p.ss[p.dim_d] + (s0 + col)));
  }
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const uint32_t r = row + 16 * i;
#pragma unroll
    for (int j = 0; j < 4; j++) tile[r][col / 2 + j] = v[i][j];
  }
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t d = d0 + 2 * lane;
  if (d >= nd) return;
#pragma unroll 4
  for (uint32_t sp = wave; sp < 64; sp += 4) {
    const uint32_t a = tile[2 * lane][sp], b = tile[2 * lane + 1][sp];
    const uint32_t sidx = s0 + 2 * sp;
    if (sidx < ns) MRL_STORE_ONCE((a & 0xffffu) | (b << 16), (uint32_t *)(dst + d_o + int64_t(sidx) * p.ds[p.dim_s] + d));
    if (sidx + 1 < ns) MRL_STORE_ONCE((a >> 16) | (b & 0xffff0000u), (uint32_t *)(dst + d_o + int64_t(sidx + 1) * p.ds[p.dim_s] + d));
  }
}

// Bytes whose source rows are whole 16-byte vectors: a 128 x 128 tile as dwords (four bytes along
// the source's contiguous dim each), loaded sixteen bytes per lane.  A lane then takes the dwords
// of four neighbouring tile rows at one column, transposes the 4 x 4 bytes in registers (byte
// permutes) and stores the four dwords into four destination rows.  The four rows are read in
// an order rotated by the lane's group, which spreads the 32 lanes of a half-wave over all banks.
__global__ __launch_bounds__(256) void k_move_tiled8v(MoveStrided p) {
  __shared__ uint32_t tile[128][33];
  uint64_t blk = blockIdx.x;
  const uint32_t ts = uint32_t(blk % p.tiles_s);
  blk /= p.tiles_s;
  const uint32_t td = uint32_t((blk + ts) % p.tiles_d);  // diagonal order, see k_move_tiled
  blk /= p.tiles_d;
  int64_t so = 0, d_o = 0;
  for (int o = int(p.rank) - 1; o >= 0; o--) {
    const uint32_t d = p.order[o];
    if (d == p.dim_s || d == p.dim_d) continue;
    const uint32_t c = uint32_t(blk % p.shape[d]);
    blk /= p.shape[d];
    so += int64_t(c) * p.ss[d], d_o += int64_t(c) * p.ds[d];
  }
  typedef uint32_t quad_t __attribute__((ext_vector_type(4)));
  const uint32_t s0 = ts * 128, d0 = td * 128, ns = p.shape[p.dim_s], nd = p.shape[p.dim_d];
  const uint8_t *src = static_cast<const uint8_t *>(p.src);
  uint8_t *dst = static_cast<uint8_t *>(p.dst);
  const uint32_t col = (threadIdx.x & 7) * 16, row = threadIdx.x >> 3;  // 8 lanes per 128-byte row
  quad_t v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t r = row + 32 * i;
    v[i] = quad_t{0, 0, 0, 0};
    if (d0 + r < nd && s0 + col < ns)
      v[i] = MRL_LOAD_ONCE((const quad_t *)(src + so + int64_t(d0 + r) * p.ss[p.dim_d] + (s0 + col)));
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t r = row + 32 * i;
#pragma unroll
    for (int j = 0; j < 4; j++) tile[r][col / 4 + j] = v[i][j];
  }
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t group = lane & 31, half = lane >> 5;  // four tile rows 4 * group .. + 3
  const uint32_t turn = group >> 3;
  const uint32_t d = d0 + 4 * group;
#pragma unroll
  for (uint32_t it = 0; it < 4; it++) {
    const uint32_t sq = it * 8 + wave * 2 + half;  // which four source bytes (one dword of a tile row)
    uint32_t x[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) x[j] = tile[4 * group + ((j + turn) & 3)][sq];
    // x[j] is tile row (j + turn) % 4: undo the rotation.
    uint32_t a[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
      const uint32_t from = (k - turn) & 3;
      a[k] = from == 0 ? x[0] : from == 1 ? x[1] : from == 2 ? x[2] : x[3];
    }
    const uint32_t lo01 = __builtin_amdgcn_perm(a[1], a[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(a[1], a[0], 0x07030602u);
    const uint32_t lo23 = __builtin_amdgcn_perm(a[3], a[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(a[3], a[2], 0x07030602u);
    const uint32_t out[4] = {__builtin_amdgcn_perm(lo23, lo01, 0x05040100u), __builtin_amdgcn_perm(lo23, lo01, 0x07060302u),
                             __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), __builtin_amdgcn_perm(hi23, hi01, 0x07060302u)};
    if (d < nd) {
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) {
        const uint32_t sidx = s0 + 4 * sq + k;
        if (sidx < ns) MRL_STORE_ONCE(out[k], (uint32_t *)(dst + d_o + int64_t(sidx) * p.ds[p.dim_s] + d));
      }
    }
  }
}

// The same for 32-bit elements that are not converted: 64 x 64 tiles, four elements (16 bytes)
// per lane on both sides.  Needs extents along both contiguous dims and all other strides in
// multiples of 4 elements and 16-byte aligned bases, so that every vector is whole and aligned.
__global__ __launch_bounds__(256) void k_move_tiled32(MoveStrided p) {
  __shared__ uint32_t tile[64][65];
  uint64_t blk = blockIdx.x;
  const uint32_t ts = uint32_t(blk % p.tiles_s);
  blk /= p.tiles_s;
  const uint32_t td = uint32_t((blk + ts) % p.tiles_d);  // diagonal order, see k_move_tiled
  blk /= p.tiles_d;
  int64_t so = 0, d_o = 0;
  for (int o = int(p.rank) - 1; o >= 0; o--) {
    const uint32_t d = p.order[o];
    if (d == p.dim_s || d == p.dim_d) continue;
    const uint32_t c = uint32_t(blk % p.shape[d]);
    blk /= p.shape[d];
    so += int64_t(c) * p.ss[d], d_o += int64_t(c) * p.ds[d];
  }
  const uint32_t col = (threadIdx.x & 15) * 4, row = threadIdx.x >> 4;  // 16 lanes per 64-element row
  const uint32_t s0 = ts * 64, d0 = td * 64, ns = p.shape[p.dim_s], nd = p.shape[p.dim_d];
  const uint32_t *src = static_cast<const uint32_t *>(p.src);
  uint32_t *dst = static_cast<uint32_t *>(p.dst);
  typedef uint32_t quad_t __attribute__((ext_vector_type(4)));
  quad_t v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t r = row + 16 * i;
    v[i] = quad_t{0, 0, 0, 0};
    if (d0 + r < nd && s0 + col < ns)
      v[i] = MRL_LOAD_ONCE((const quad_t *)(src + so + int64_t(d0 + r) * p.ss[p.dim_d] + (s0 + col)));
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t r = row + 16 * i;
    tile[r][col] = v[i][0], tile[r][col + 1] = v[i][1], tile[r][col + 2] = v[i][2], tile[r][col + 3] = v[i][3];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t r = row + 16 * i;
    if (s0 + r < ns && d0 + col < nd) {
      const quad_t out{tile[col][r], tile[col + 1][r], tile[col + 2][r], tile[col + 3][r]};
      __builtin_nontemporal_store(out, (quad_t *)(dst + d_o + int64_t(s0 + r) * p.ds[p.dim_s] + (d0 + col)));
    }
  }
}

// Both sides contiguous along the same digit, in whole vectors of V elements (shape, strides and
// extents count vectors; the wider side of a vector is 16, 8 or 4 bytes), converted or not.  Bound
// by memory, so what matters is the order: a workgroup's tile is long along the digit that
// continues the destination's runs AND along the one that continues the source's, so that both
// sides see whole cache lines (f32 2048 x 16384 into bf16 strips of 16 columns, runs of 64 and
// 32 bytes: an element per thread in destination order 133 us, this 42).  UNROLL vectors a
// thread, their loads in flight together.
constexpr int MOVE_RUNS_ACT = 4;   // digits a tile extends along at most
template <int SE, int DE, int V, int UNROLL, bool DIAGONAL = false>
__global__ __launch_bounds__(256) void k_move_runs(MoveTile p) {
  int64_t base_s, base_d;
  uint32_t room[MOVE_MAX_RANK];
  tile_origin<DIAGONAL>(p, base_s, base_d, room);
  uint32_t raw[UNROLL][V], to[UNROLL];
  bool inside[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; u++) {
    uint32_t rem = threadIdx.x + u * 256, so = 0;
    inside[u] = rem < p.tile;
    to[u] = 0;
#pragma unroll
    for (int d = 0; d < MOVE_RUNS_ACT; d++) {
      const uint32_t rest = div_small(rem, p.ext[d], p.inv_ext[d]), c = rem - rest * p.ext[d];
      rem = rest;
      inside[u] = inside[u] && c < room[d];
      so += c * uint32_t(p.ss[d]), to[u] += c * uint32_t(p.ds[d]);
    }
    // (a vector outside the tensor loads the tile's first one instead: no branch between the loads)
    load_run<SE, V>(p.src, (base_s + (inside[u] ? so : 0u)) * V, raw[u]);
  }
  with_dtypes<SE, DE>(p.sdt, p.ddt, [&](auto sd, auto dd) {
#pragma unroll
    for (int u = 0; u < UNROLL; u++)
#pragma unroll
      for (int e = 0; e < V; e++) raw[u][e] = convert_raw(raw[u][e], decltype(sd)::value, decltype(dd)::value);
  });
#pragma unroll
  for (int u = 0; u < UNROLL; u++)
    if (inside[u]) store_run<DE, V>(p.dst, (base_d + to[u]) * V, raw[u]);
}
// Without tiles, a vector a thread in destination order: a tile's arithmetic, a dozen digits of its origin ahead
// of the first load, is 1 to 3 us of a launch (launch_move_view says where they are earned back).
template <int SE, int DE, int V>
__global__ __launch_bounds__(256) void k_move_runs(MoveStrided p) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.count) return;
  int64_t so, d_o;
  place_of(p, i, so, d_o);
  uint32_t raw[V];
  load_run<SE, V>(p.src, so * V, raw);
  with_dtypes<SE, DE>(p.sdt, p.ddt, [&](auto sd, auto dd) {
#pragma unroll
    for (int e = 0; e < V; e++) raw[e] = convert_raw(raw[e], decltype(sd)::value, decltype(dd)::value);
  });
  store_run<DE, V>(p.dst, d_o * V, raw);
}

// Without a tile, an element a thread in destination order: small tensors, as above.
template <int SE, int DE>
__global__ __launch_bounds__(256) void k_move_gather(MoveStrided p) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= p.count) return;
  int64_t so, d_o;
  place_of(p, i, so, d_o);
  uint32_t raw = load_sized<SE>(p.src, so);
  with_dtypes<SE, DE>(p.sdt, p.ddt, [&](auto sd, auto dd) { raw = convert_raw(raw, decltype(sd)::value, decltype(dd)::value); });
  store_sized<DE>(p.dst, d_o, raw);
}

// Four 16-byte vectors per thread in flight, streamed past the caches: 6.5 TB/s on a 256 MiB
// copy against 5.7 TB/s for one cached vector per thread.
constexpr int COPY_UNROLL = 4;
typedef unsigned v4u __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_copy16(const v4u *__restrict__ src, v4u *__restrict__ dst,
                                                uint64_t vecs) {
  const uint64_t step = uint64_t(gridDim.x) * 256 * COPY_UNROLL;
  for (uint64_t i = uint64_t(blockIdx.x) * 256 * COPY_UNROLL + threadIdx.x; i < vecs; i += step) {
    v4u v[COPY_UNROLL];
#pragma unroll
    for (int u = 0; u < COPY_UNROLL; u++)
      if (i + u * 256 < vecs) v[u] = MRL_LOAD_ONCE(src + i + u * 256);
#pragma unroll
    for (int u = 0; u < COPY_UNROLL; u++)
      if (i + u * 256 < vecs) __builtin_nontemporal_store(v[u], dst + i + u * 256);
  }
}

// bf16 -> f32 of a whole buffer, position by position (exact: a 16-bit shift).
__global__ __launch_bounds__(256) void k_widen_bf16(const uint16_t *__restrict__ src, uint32_t *__restrict__ dst,
                                                    uint64_t count) {
  const uint64_t step = uint64_t(gridDim.x) * blockDim.x;
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += step)
    dst[i] = uint32_t(src[i]) << 16;
}

// Copies [batch][rows][cols] with contiguous rows, starting on any element, into `dst_rows` rows of whole
// 16-byte chunks, zeros from each row's end on and in the rows past the last.  A thread makes one or four
// chunks, each out of the two aligned chunks of the source it lies in (with a load per element, u8
// 5440 x 1683 x 2556 took 62.9 us in all; 46.7 now).
struct PadJob {
  const uint8_t *src;
  chunk_t *dst;
  uint64_t row_bytes;                     // of a source row
  uint32_t rows, dst_rows, row_chunks;    // row_chunks: of a destination row
  uint32_t chunks;                        // destination chunks in all
  int64_t src_batch, src_ld;                        // bytes
  FastDiv by_row_chunks, by_dst_rows;
  uint32_t panel_chunks;                  // of a row of a panel (0: no panels)
  FastDiv by_panel_chunks;
};
constexpr int PAD_UNROLL = 4;
template <int UNROLL>
__device__ inline void pad_chunks(const PadJob &j) {
  const uint32_t first = blockIdx.x * (256 * UNROLL) + threadIdx.x;
  chunk_t lo[UNROLL], hi[UNROLL];
  int left[UNROLL];
  uint32_t shift[UNROLL], to[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; u++) {
    const uint32_t i = min(first + u * 256, j.chunks - 1);
    const uint32_t line = j.by_row_chunks.div(i), entry = j.by_dst_rows.div(line), row = line - entry * j.dst_rows;
    const PadChunk c = pad_chunk(i - line * j.row_chunks, row < j.rows ? j.row_bytes : 0);
    left[u] = c.left;
    to[u] = i;
    if (j.panel_chunks != 0) {
      const uint32_t in_row = i - line * j.row_chunks, panel = j.by_panel_chunks.div(in_row);
      to[u] = (entry * j.row_chunks + panel * j.panel_chunks) * j.dst_rows + row * j.panel_chunks + in_row - panel * j.panel_chunks;
    }
    // (a chunk with nothing in it reads the row's first instead)
    const uint8_t *from = j.src + int64_t(entry) * j.src_batch + int64_t(min(row, j.rows - 1)) * j.src_ld + c.at;
    shift[u] = uint32_t(uintptr_t(from) & 15);
    from -= shift[u];
    lo[u] = *(const chunk_t *)from;
    hi[u] = *(const chunk_t *)(from + (int(shift[u]) + left[u] > 16 ? 16 : 0));
  }
#pragma unroll
  for (int u = 0; u < UNROLL; u++)
    if (first + u * 256 < j.chunks) j.dst[to[u]] = keep_bytes(cut_chunk(lo[u], hi[u], shift[u]), left[u]);
}
template <int UNROLL>
__global__ __launch_bounds__(256) void k_pad_rows(PadJob j) { pad_chunks<UNROLL>(j); }
// Two such copies in one launch (blockIdx.y names the copy): the two operands of a Matmul whose rows
// are not whole 16-byte chunks each took a launch of about 2.4 us for their padded copy (int8 1000^3).
template <int UNROLL>
__global__ __launch_bounds__(256) void k_pad_rows_pair(PadJob j0, PadJob j1) {
  const PadJob &j = blockIdx.y ? j1 : j0;
  if (blockIdx.x * (256 * UNROLL) < j.chunks) pad_chunks<UNROLL>(j);
}

__global__ void k_copy1(const uint8_t *src, uint8_t *dst, uint64_t bytes) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < bytes) dst[i] = src[i];
}

// -------------------------------------------------------------------- matmul
struct MM {
  const void *a, *b;
  void *c;
  int dta, dtb, dtc;
  uint32_t B, M, K, N;
  int64_t sa[3], sb[3], sc[3];
  int accum;
};

template <bool FLOAT_OUT>
__global__ __launch_bounds__(256) void k_matmul_generic(MM p) {
  __shared__ uint32_t ta[16][17], tb[16][17];
  const uint32_t tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  // One 16 x 16 output tile per workgroup, tiles numbered n-fastest, then m, then batch, in
  // grid.x alone (grid.y and grid.z stop at 65535, which 2^20 rows would pass).
  const uint32_t tiles_n = (p.N + 15) / 16, tiles_m = (p.M + 15) / 16;
  const uint32_t tile_j = blockIdx.x % tiles_n, tile_i = (blockIdx.x / tiles_n) % tiles_m;
  const uint32_t bi = blockIdx.x / tiles_n / tiles_m;
  const uint32_t j = tile_j * 16 + tx, i = tile_i * 16 + ty;
  const bool live = i < p.M && j < p.N;
  const int64_t coff = int64_t(bi) * p.sc[0] + int64_t(i) * p.sc[1] + int64_t(j) * p.sc[2];
  float facc = 0.0f;
  uint32_t iacc = 0;
  if (p.accum && live) {
    if (FLOAT_OUT) facc = ((const float *)p.c)[coff];
    else iacc = load_u32(p.c, p.dtc, coff, MRL_U32);
  }
  for (uint32_t k0 = 0; k0 < p.K; k0 += 16) {
    {  // A tile: row i, col k0+tx ; B tile: row k0+ty, col j
      const uint32_t ka = k0 + tx, kb = k0 + ty;
      uint32_t av = 0, bv = 0;
      if (i < p.M && ka < p.K) {
        const int64_t o = int64_t(bi) * p.sa[0] + int64_t(i) * p.sa[1] + int64_t(ka) * p.sa[2];
        av = FLOAT_OUT ? __float_as_uint(load_f32(p.a, p.dta, o)) : load_u32(p.a, p.dta, o, p.dtc);
      }
      if (kb < p.K && j < p.N) {
        const int64_t o = int64_t(bi) * p.sb[0] + int64_t(kb) * p.sb[1] + int64_t(j) * p.sb[2];
        bv = FLOAT_OUT ? __float_as_uint(load_f32(p.b, p.dtb, o)) : load_u32(p.b, p.dtb, o, p.dtc);
      }
      ta[ty][tx] = av;
      tb[ty][tx] = bv;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t kk = 0; kk < 16; kk++) {
      if (FLOAT_OUT) facc += __uint_as_float(ta[ty][kk]) * __uint_as_float(tb[kk][tx]);
      else iacc += ta[ty][kk] * tb[kk][tx];
    }
    __syncthreads();
  }
  if (live) {
    if (FLOAT_OUT) ((float *)p.c)[coff] = facc;
    else store_u32(p.c, p.dtc, coff, iacc);
  }
}

// ---------------------------------------------------------------------- conv
struct CV {
  const void *img, *filt;
  void *out;
  int dti, dtf, dto;
  uint32_t B, F, C, OH, OW, FH, FW;
  int64_t si[4], sf[4], so[4];
  int accum;
};

template <bool FLOAT_OUT>
__global__ __launch_bounds__(256) void k_conv_generic(CV p) {
  const uint64_t total = uint64_t(p.B) * p.F * p.OH * p.OW;
  const uint64_t idx = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  // Decode with f fastest so that NHWC outputs are written contiguously.
  uint64_t r = idx;
  const uint32_t f = uint32_t(r % p.F); r /= p.F;
  const uint32_t x = uint32_t(r % p.OW); r /= p.OW;
  const uint32_t y = uint32_t(r % p.OH); r /= p.OH;
  const uint32_t b = uint32_t(r);
  const int64_t ooff = b * p.so[0] + f * p.so[1] + y * p.so[2] + x * p.so[3];
  float facc = 0.0f;
  uint32_t iacc = 0;
  if (p.accum) {
    if (FLOAT_OUT) facc = ((const float *)p.out)[ooff];
    else iacc = load_u32(p.out, p.dto, ooff, MRL_U32);
  }
  for (uint32_t c = 0; c < p.C; c++)
    for (uint32_t rr = 0; rr < p.FH; rr++)
      for (uint32_t s = 0; s < p.FW; s++) {
        const int64_t io = b * p.si[0] + c * p.si[1] + int64_t(y + rr) * p.si[2] + int64_t(x + s) * p.si[3];
        const int64_t fo = f * p.sf[0] + c * p.sf[1] + rr * p.sf[2] + s * p.sf[3];
        if (FLOAT_OUT) facc += load_f32(p.img, p.dti, io) * load_f32(p.filt, p.dtf, fo);
        else iacc += load_u32(p.img, p.dti, io, p.dto) * load_u32(p.filt, p.dtf, fo, p.dto);
      }
  if (FLOAT_OUT) ((float *)p.out)[ooff] = facc;
  else store_u32(p.out, p.dto, ooff, iacc);
}

// The same with one wavefront per output element, its lanes striding over the C * FH * FW
// products: for a handful of outputs with a long reduction (examples/simple_conv_x86.rs: 8 outputs
// of 72 products each) the one-thread-per-output kernel is a chain of dependent loads.
template <bool FLOAT_OUT>
__global__ __launch_bounds__(256) void k_conv_generic_wave(CV p) {
  const uint64_t total = uint64_t(p.B) * p.F * p.OH * p.OW;
  const uint64_t idx = uint64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (idx >= total) return;
  const uint32_t lane = threadIdx.x & 63;
  uint64_t r = idx;
  const uint32_t f = uint32_t(r % p.F); r /= p.F;
  const uint32_t x = uint32_t(r % p.OW); r /= p.OW;
  const uint32_t y = uint32_t(r % p.OH); r /= p.OH;
  const uint32_t b = uint32_t(r);
  const int64_t ooff = b * p.so[0] + f * p.so[1] + y * p.so[2] + x * p.so[3];
  float facc = 0.0f;
  uint32_t iacc = 0;
  const uint32_t window = p.FH * p.FW, terms = p.C * window;
  for (uint32_t t = lane; t < terms; t += 64) {
    const uint32_t c = t / window, rr = (t % window) / p.FW, s = t % p.FW;
    const int64_t io = b * p.si[0] + c * p.si[1] + int64_t(y + rr) * p.si[2] + int64_t(x + s) * p.si[3];
    const int64_t fo = f * p.sf[0] + c * p.sf[1] + rr * p.sf[2] + s * p.sf[3];
    if (FLOAT_OUT) facc += load_f32(p.img, p.dti, io) * load_f32(p.filt, p.dtf, fo);
    else iacc += load_u32(p.img, p.dti, io, p.dto) * load_u32(p.filt, p.dtf, fo, p.dto);
  }
  for (int o = 32; o > 0; o >>= 1) {
    facc += __shfl_xor(facc, o);
    iacc += uint32_t(__shfl_xor(int(iacc), o));
  }
  if (lane != 0) return;
  if (p.accum) {
    if (FLOAT_OUT) facc += ((const float *)p.out)[ooff];
    else iacc += load_u32(p.out, p.dto, ooff, MRL_U32);
  }
  if (FLOAT_OUT) ((float *)p.out)[ooff] = facc;
  else store_u32(p.out, p.dto, ooff, iacc);
}

// ------------------------------------------------------------------- softmax
// One wavefront per line along an arbitrary-stride scan dim: max, then exp and sum, then
// divide (morello/src/verification.rs:166-184).
struct SM {
  const float *in;
  float *out;
  uint32_t rank, scan_dim;
  uint32_t shape[MRL_MAX_RANK];
  int64_t si[MRL_MAX_RANK], so[MRL_MAX_RANK];
  uint64_t lines;
};

__device__ inline float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}
__device__ inline float wave_sum(float v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__global__ __launch_bounds__(256) void k_softmax_generic(SM p) {
  const uint64_t line = uint64_t(blockIdx.x) * 4 + threadIdx.x / 64;
  const uint32_t lane = threadIdx.x % 64;
  if (line >= p.lines) return;
  uint64_t r = line;
  int64_t ibase = 0, obase = 0;
  for (int d = int(p.rank) - 1; d >= 0; d--) {
    if (uint32_t(d) == p.scan_dim) continue;
    const uint32_t c = uint32_t(r % p.shape[d]);
    r /= p.shape[d];
    ibase += c * p.si[d];
    obase += c * p.so[d];
  }
  const uint32_t n = p.shape[p.scan_dim];
  const int64_t is = p.si[p.scan_dim], os = p.so[p.scan_dim];
  float mx = -3.40282347e+38f;
  bool nan = false;
  for (uint32_t i = lane; i < n; i += 64) {
    const float v = p.in[ibase + i * is];
    nan |= v != v;
    mx = fmaxf(mx, v);
  }
  mx = wave_max(mx);
  if (__any(nan)) mx = __uint_as_float(0x7fc00000u);
  float sum = 0.0f;
  for (uint32_t i = lane; i < n; i += 64) {
    const float e = expf(p.in[ibase + i * is] - mx);
    p.out[obase + i * os] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  for (uint32_t i = lane; i < n; i += 64) p.out[obase + i * os] /= sum;
}

// The scan dim is strided but another dim (`fast`) is contiguous on both sides: a workgroup
// takes 64 consecutive positions of `fast` (one per lane, so every access is a 256-byte run)
// and its WAVES waves (16 for long scan dims) split the scan dim; each lane keeps the online (max, denominator) pair of
// morello/src/spec.rs:96-106 over its share, the shares are merged through LDS with the
// parts formula (spec.rs:107-132), and a second sweep writes exp(x - max) / denominator.
// With few columns (fewer workgroups than compute units) the scan dim is also cut into `chunks`
// pieces of chunk_len steps, blockIdx.y naming the piece, and the work into two launches
// (morello/src/scheduling/parallel_softmax.rs:24-223 on the GPU's grid): PHASE 1 leaves every
// piece's pair in `pairs` ([column tile][piece][lane]), PHASE 2 merges a column's pairs and writes
// its own piece.  PHASE 0 is the whole Softmax in one launch.
struct SMC {
  SM s;
  uint32_t fast, fast_tiles;
  uint32_t chunks, chunk_len;
  float2 *pairs;
};
// exp(x) for x <= 0 (and NaN) as 2^t (one instruction at a quarter of the vector rate) with t = x log2(e)
// formed in two parts, the low part applied as a first-order factor: within two units in the last
// place, where libm's expf costs about twenty instructions.  The column kernel is bound by those:
// 2048 x 4096 over dim 0 took 27 us with expf.  Arguments below -150 give 0 like anything below -104.
__device__ inline float exp_nonpositive(float x) {
  x = x < -150.0f ? -150.0f : x;
  const float t = x * 1.44269504f;
  const float lo = __builtin_fmaf(x, 1.44269504f, -t) + x * 1.92596299e-8f;
  return __builtin_amdgcn_exp2f(t) * __builtin_fmaf(lo, 0.693147181f, 1.0f);
}
__device__ inline void merge_pair(float &m, float &d, float om, float od) {
  const float nm = (om != om || m != m) ? __uint_as_float(0x7fc00000u) : fmaxf(m, om);
  d = d * expf(m - nm) + od * expf(om - nm);
  m = nm;
}
// A scan dim of at most 16 elements beside a contiguous dim: a thread per column, the column in
// registers, 256 consecutive columns per workgroup (q.fast_tiles counts tiles of 256 here).  The
// kernel below would give each handful of rows a workgroup of its own, with its start-up and its
// exchange through LDS: 8 x 8 x 1024 x 1024 over dim 1 took 295 us that way.
__global__ __launch_bounds__(256) void k_softmax_cols_short(SMC q) {
  const SM &p = q.s;
  uint64_t r = blockIdx.x;
  const uint32_t f = uint32_t(r % q.fast_tiles) * 256 + threadIdx.x;
  r /= q.fast_tiles;
  int64_t ibase = 0, obase = 0;
  for (int d = int(p.rank) - 1; d >= 0; d--) {
    if (uint32_t(d) == p.scan_dim || uint32_t(d) == q.fast) continue;
    const uint32_t c = uint32_t(r % p.shape[d]);
    r /= p.shape[d];
    ibase += c * p.si[d];
    obase += c * p.so[d];
  }
  if (f >= p.shape[q.fast]) return;
  ibase += f, obase += f;  // unit stride on both sides
  const uint32_t n = p.shape[p.scan_dim];
  const int64_t is = p.si[p.scan_dim], os = p.so[p.scan_dim];
  float x[16];
  float m = -3.40282347e+38f;
  bool nan = false;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    x[j] = uint32_t(j) < n ? p.in[ibase + j * is] : -3.40282347e+38f;
    nan |= x[j] != x[j];
    m = fmaxf(m, x[j]);
  }
  if (nan) m = __uint_as_float(0x7fc00000u);
  float den = 0.0f;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    x[j] = exp_nonpositive(x[j] - m);
    den += uint32_t(j) < n ? x[j] : 0.0f;
  }
  const float inv = 1.0f / den;
#pragma unroll
  for (int j = 0; j < 16; j++)
    if (uint32_t(j) < n) MRL_STORE_ONCE(x[j] * inv, p.out + obase + j * os);
}

// R: not 0 where the scan dim is at most WAVES * R: PHASE 0 then keeps the columns in registers, R values a lane, and
// reads each element once.  Bound by memory; over dim 1, us before -> now: 25 x 370 x 961 30.4 -> 23.5, 20 x 200 x 2000 20.7 -> 14.1,
// 64 x 60 x 1000 10.1 -> 7.2, 6 x 120 x 135 13.1 -> 5.7.
// RUNS: an XCD takes neighbouring tiles, which share the lines that rows of odd lengths cross, in its L2 (us, dealt over the XCDs / in runs: 16 x 1793 x 673 68.4 /
// 51.3, 20 x 1500 x 700 65.4 / 52.8, 32 x 513 x 1000 40.6 / 33.0).  Rows of whole lines that are read twice are dealt over the XCDs (24 x 1160 x 2752 167 / 170, 6 x
// 3000 x 4000 160 / 165).
template <int WAVES, int PHASE, int R = 0, bool RUNS = (R > 0)>
__global__ __launch_bounds__(64 * WAVES) void k_softmax_cols(SMC q) {
  const SM &p = q.s;
  __shared__ float sm_max[WAVES][64], sm_den[WAVES][64];
  const uint32_t lane = threadIdx.x % 64, w = threadIdx.x / 64;
  uint64_t r = RUNS ? xcd_run(blockIdx.x, gridDim.x) : blockIdx.x;
  const uint32_t f = uint32_t(r % q.fast_tiles) * 64 + lane;
  r /= q.fast_tiles;
  int64_t ibase = 0, obase = 0;
  for (int d = int(p.rank) - 1; d >= 0; d--) {
    if (uint32_t(d) == p.scan_dim || uint32_t(d) == q.fast) continue;
    const uint32_t c = uint32_t(r % p.shape[d]);
    r /= p.shape[d];
    ibase += c * p.si[d];
    obase += c * p.so[d];
  }
  const bool live = f < p.shape[q.fast];
  ibase += f, obase += f;  // unit stride on both sides
  const uint32_t first = PHASE == 0 ? 0 : blockIdx.y * q.chunk_len;
  const uint32_t n = PHASE == 0 ? p.shape[p.scan_dim] : min(p.shape[p.scan_dim], first + q.chunk_len);
  const int64_t is = p.si[p.scan_dim], os = p.so[p.scan_dim];
  constexpr int UNROLL = 8;
  float m, d;
  if constexpr (R > 0) {
    // All loads go out before the first is looked at; a step past the end is the last one again, a column past the end the last one.
    const float *from = p.in + ibase - (live ? 0 : f - (p.shape[q.fast] - 1));
    float x[R];
    float mx = -3.40282347e+38f, den = 0.0f;
    bool nan = false;
#pragma unroll
    for (int j = 0; j < R; j++) x[j] = from[min(w + j * WAVES, n - 1) * is];
#pragma unroll
    for (int j = 0; j < R; j++) nan |= x[j] != x[j], mx = fmaxf(mx, x[j]);
    sm_max[w][lane] = nan ? __uint_as_float(0x7fc00000u) : mx;
    __syncthreads();
    m = sm_max[0][lane];
#pragma unroll
    for (int o = 1; o < WAVES; o++) {
      const float other = sm_max[o][lane];
      m = other != other || m != m ? __uint_as_float(0x7fc00000u) : fmaxf(m, other);
    }
#pragma unroll
    for (int j = 0; j < R; j++) {
      x[j] = exp_nonpositive(x[j] - m);
      den += w + j * WAVES < n ? x[j] : 0.0f;
    }
    sm_den[w][lane] = den;
    __syncthreads();
    d = 0.0f;
#pragma unroll
    for (int o = 0; o < WAVES; o++) d += sm_den[o][lane];
    const float inv = 1.0f / d;
    if (live)
#pragma unroll
      for (int j = 0; j < R; j++)
        if (w + j * WAVES < n) MRL_STORE_ONCE(x[j] * inv, p.out + obase + int64_t(w + j * WAVES) * os);
    return;
  }
  if (PHASE != 2) {
    float mx = -3.40282347e+38f, den = 0.0f;
    bool nan = false;
    // Eight loads in flight per lane, then one rescale of the running denominator for the eight.
    if (live)
      for (uint32_t i0 = first + w; i0 < n; i0 += WAVES * UNROLL) {
        float x[UNROLL];
        float nm = mx;
#pragma unroll
        for (int j = 0; j < UNROLL; j++) {
          const uint32_t i = i0 + j * WAVES;
          x[j] = i < n ? p.in[ibase + i * is] : -3.40282347e+38f;
          nan |= x[j] != x[j];
          nm = fmaxf(nm, x[j]);
        }
        float add = 0.0f;
#pragma unroll
        for (int j = 0; j < UNROLL; j++) add += i0 + j * WAVES < n ? exp_nonpositive(x[j] - nm) : 0.0f;
        den = den * exp_nonpositive(mx - nm) + add;
        mx = nm;
      }
    if (nan) mx = __uint_as_float(0x7fc00000u);
    sm_max[w][lane] = mx, sm_den[w][lane] = den;
    __syncthreads();
    m = sm_max[0][lane], d = sm_den[0][lane];
#pragma unroll
    for (int o = 1; o < WAVES; o++) merge_pair(m, d, sm_max[o][lane], sm_den[o][lane]);
    if (PHASE == 1) {
      if (w == 0) q.pairs[(uint64_t(blockIdx.x) * q.chunks + blockIdx.y) * 64 + lane] = make_float2(m, d);
      return;
    }
  } else {
    // The column's pairs: every wave merges its share of the pieces, eight loads in flight at a
    // time, and the waves' results meet in LDS.
    const float2 *mine = q.pairs + uint64_t(blockIdx.x) * q.chunks * 64 + lane;
    m = -3.40282347e+38f, d = 0.0f;
    for (uint32_t c0 = w; c0 < q.chunks; c0 += WAVES * UNROLL) {
      float2 pc[UNROLL];
#pragma unroll
      for (int j = 0; j < UNROLL; j++) {
        const uint32_t c = c0 + j * WAVES;
        pc[j] = c < q.chunks ? mine[uint64_t(c) * 64] : make_float2(-3.40282347e+38f, 0.0f);
      }
#pragma unroll
      for (int j = 0; j < UNROLL; j++) merge_pair(m, d, pc[j].x, pc[j].y);
    }
    sm_max[w][lane] = m, sm_den[w][lane] = d;
    __syncthreads();
    m = sm_max[0][lane], d = sm_den[0][lane];
#pragma unroll
    for (int o = 1; o < WAVES; o++) merge_pair(m, d, sm_max[o][lane], sm_den[o][lane]);
  }
  const float inv_d = 1.0f / d;
  if (live)
    for (uint32_t i0 = first + w; i0 < n; i0 += WAVES * UNROLL) {
      float x[UNROLL];
#pragma unroll
      for (int j = 0; j < UNROLL; j++) {
        const uint32_t i = i0 + j * WAVES;
        x[j] = i < n ? p.in[ibase + i * is] : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < UNROLL; j++) {
        const uint32_t i = i0 + j * WAVES;
        if (i < n) MRL_STORE_ONCE(exp_nonpositive(x[j] - m) * inv_d, p.out + obase + i * os);
      }
    }
}

__global__ void k_fill_zero(uint32_t *p, uint64_t words, uint8_t *tail, uint32_t tail_bytes) {
  const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint64_t step = uint64_t(gridDim.x) * blockDim.x;
  for (uint64_t w = i; w < words; w += step) p[w] = 0;
  if (i < tail_bytes) tail[i] = 0;
}

bool float_out(int dt) { return dt == MRL_F32; }

}  // namespace

hipError_t launch_relayout(const void *src, void *dst, const LayoutEval &sl, const LayoutEval &dl,
                           uint32_t es, uint64_t count, hipStream_t stream) {
  if (count == 0) return hipSuccess;
  const uint32_t blocks = uint32_t((count + 255) / 256);
  plan::work(plan::UNIT_VALU, 40.0 * count, 2.0 * count * es);  // index arithmetic per element
  MRL_LAUNCH(k_relayout, dim3(blocks), dim3(256), 0, stream, (const uint8_t *)src,
                     (uint8_t *)dst, sl, dl, es, count);
  return mrl::plan::last_error();
}

hipError_t launch_move_generic(const void *src, void *dst, const LayoutEval &sl, const LayoutEval &dl,
                               int sdt, int ddt, uint64_t count, hipStream_t stream) {
  if (count == 0) return hipSuccess;
  const uint32_t blocks = uint32_t((count + 255) / 256);
  plan::work(plan::UNIT_VALU, 40.0 * count, double(count) * (mrl_dtype_size(sdt) + mrl_dtype_size(ddt)));
  MRL_LAUNCH(k_move_generic, dim3(blocks), dim3(256), 0, stream, src, dst, sl, dl, sdt, ddt, count);
  return mrl::plan::last_error();
}

hipError_t launch_copy(const void *src, void *dst, uint64_t bytes, hipStream_t stream) {
  const uint64_t vecs = bytes / 16, tail = bytes % 16;
  if (vecs) {
    uint64_t blocks = (vecs + 256 * COPY_UNROLL - 1) / (256 * COPY_UNROLL);
    if (blocks > 8192) blocks = 8192;  // grid-stride: 32 blocks per CU on a 256-CU part
    plan::work(plan::UNIT_STREAM, 0, 2.0 * bytes);
    MRL_LAUNCH(k_copy16, dim3(uint32_t(blocks)), dim3(256), 0, stream, (const v4u *)src,
                       (v4u *)dst, vecs);
  }
  if (tail)
    MRL_LAUNCH(k_copy1, dim3(1), dim3(16), 0, stream, (const uint8_t *)src + vecs * 16,
                       (uint8_t *)dst + vecs * 16, tail);
  return mrl::plan::last_error();
}

namespace {
// Up to this many elements a Move with nothing to vectorise runs an element per thread: one round
// of workgroups whatever the layouts, where the tiled kernels' loops over a handful of tiles take
// three times as long.
constexpr uint64_t MOVE_TINY = 65536;
// Up to this many an element or a vector a thread in destination order, no tiles: scattered reads come out of
// the caches, and a tile's arithmetic is what is left.  Over 1200 random layouts of up to five dims (geometric means, tiles /
// without): 64 to 128 thousand elements 4.8 / 3.2 us, 512 thousand to 1 Mi 6.4 / 4.8 (vectors 4.9 / 4.5), 2 to 4 Mi 9.7 / 12.6
// (6.5 / 10.8); [45, 1963, 4] to [45, 4, 1963] f32 5.8 / 4.3, bf16 5.0 / 3.3.  Between 1 and 2 Mi it is either, by layout.
constexpr uint64_t MOVE_SMALL = 1u << 20;
// Whole 16-byte vectors in runs of 64 bytes or more, nothing converted: either side then reads and writes half a cache
// line at least in any order, and tiles pay later (4 to 8 MB 5.8 / 3.8 us, 8 to 16 MB 5.4 / 4.5, 16 to 32 MB 7.6 / 7.2 but up to 25 % either way, 32 to 64 MB 15.4 / 17.7).
constexpr uint64_t MOVE_DIRECT_BYTES = 16u << 20;

// A MoveTile's per-digit arrays from a view and the tile's extents.  `first`: digits in the order a
// vector's number counts them (k_move_runs), nullptr for any order with the extended digits first.
void fill_tile(MoveTile *t, const MoveStrided &p, const uint32_t *ext, const uint32_t *tstride_s, const uint32_t *tstride_d,
               const uint32_t *first, uint32_t *n_act, uint64_t *blocks) {
  auto inverse = [](uint32_t x) { return x <= 1 ? 0u : uint32_t(((uint64_t(1) << 32) + x - 1) / x); };
  t->src = p.src, t->dst = p.dst, t->sdt = p.sdt, t->ddt = p.ddt;
  uint32_t perm[MOVE_MAX_RANK], n = 0;
  bool taken[MOVE_MAX_RANK] = {};
  for (uint32_t i = 0; first && i < *n_act; i++) perm[n++] = first[i], taken[first[i]] = true;
  for (int extended = 1; extended >= 0; extended--) {
    for (uint32_t d = 0; d < MOVE_MAX_RANK; d++)
      if (!taken[d] && (ext[d] > 1) == bool(extended)) perm[n++] = d, taken[d] = true;
    if (extended && !first) *n_act = n;
  }
  *blocks = 1;
  for (uint32_t i = 0; i < MOVE_MAX_RANK; i++) {
    const uint32_t d = perm[i];
    t->shape[i] = p.shape[d], t->ss[i] = p.ss[d], t->ds[i] = p.ds[d], t->ext[i] = ext[d];
    t->chunks[i] = (p.shape[d] + ext[d] - 1) / ext[d], t->by_chunks[i] = FastDiv(t->chunks[i]);
    t->inv_ext[i] = inverse(ext[d]);
    t->tstride_s[i] = tstride_s ? tstride_s[d] : 1, t->tstride_d[i] = tstride_d ? tstride_d[d] : 1;
    t->inv_s[i] = inverse(t->tstride_s[i]), t->inv_d[i] = inverse(t->tstride_d[i]);
    *blocks *= t->chunks[i];
  }
}

// k_move_runs' tile over a view whose shared digit counts vectors of `vec` elements: how many vectors it
// holds, and how many tiles there are.  0 where it would have more workgroups than a launch takes.
uint32_t runs_tile(const MoveStrided &p, uint32_t shared, uint32_t vec, uint32_t se, uint32_t de, MoveTile *t, uint64_t *blocks) {
  const uint32_t rank = p.rank;
  // Four vectors a thread once every compute unit gets two such workgroups.
  const uint32_t tile_cap = p.count >= 1024ull * 2 * g_compute_units ? 1024 : 256;
  uint32_t ext[MOVE_MAX_RANK], first[MOVE_RUNS_ACT], n_first = 0, tile = 1;
  for (uint32_t d = 0; d < MOVE_MAX_RANK; d++) ext[d] = 1;
  auto known = [&](uint32_t d) { return std::find(first, first + n_first, d) != first + n_first; };
  auto take = [&](uint32_t d, uint32_t most) {
    const uint32_t e = std::min({p.shape[d], most, tile_cap / tile});
    if (e <= 1 || known(d) || n_first == MOVE_RUNS_ACT) return;
    first[n_first++] = d, ext[d] = e, tile *= e;
  };
  // (a shared digit longer than 256 vectors is cut into even pieces)
  take(shared, p.shape[shared] <= 256 ? 256u : (p.shape[shared] + (p.shape[shared] + 255) / 256 - 1) / ((p.shape[shared] + 255) / 256));
  auto next = [&](const int64_t *stride, int behind) {   // the digit that continues the runs of one side
    int best = -1;
    for (uint32_t d = 0; d < rank; d++)
      if (d != shared && int(d) != behind && p.shape[d] > 1 && (behind < 0 || stride[d] >= stride[behind]) &&
          (best < 0 || stride[d] < stride[best]))
        best = int(d);
    return best;
  };
  const int next_d = next(p.ds, -1), next_s = next(p.ss, -1);
  if (next_d >= 0 && next_s >= 0 && next_s != next_d) {
    // 512 bytes of the source side, along two digits if need be, the rest of the tile along the destination's (of 32 a vector from rows 32 KiB
    // apart 1 KiB: f32 2048 x 16384 into bf16 strips of 16 43.9 / 42.0 us, 8192 x 8192 87.2 / 81.1; but 4096 x 4096 18.8 / 20.5)
    const uint32_t piece = vec * se == 32 && p.ss[next_d] * int64_t(vec * se) >= 32768 ? 1024 : 512;
    const uint32_t want_s = std::min(std::max(1u, piece / (ext[shared] * vec * se)), std::max(1u, tile_cap / tile));
    const int further = p.shape[next_s] < want_s ? next(p.ss, next_s) : -1;
    const bool two = further >= 0 && further != next_d;
    const uint32_t s1 = std::min(want_s, p.shape[next_s]), s2 = two ? std::min(want_s / s1, p.shape[further]) : 1;
    take(uint32_t(next_d), std::max(1u, tile_cap / tile / (s1 * s2)));
    take(uint32_t(next_s), p.shape[next_s]);
    if (two) take(uint32_t(further), p.shape[further]);
  } else if (next_d >= 0) {
    take(uint32_t(next_d), p.shape[next_d]);
  }
  // What is left of the tile: along the destination's further digits, or, when they come to the tile's last
  // digit, along the longest.
  for (int o = int(rank) - 1; o >= 0 && n_first + 1 < uint32_t(MOVE_RUNS_ACT); o--) take(p.order[o], p.shape[p.order[o]]);
  int longest = -1;
  for (uint32_t d = 0; d < rank; d++)
    if (!known(d) && (longest < 0 || p.shape[d] > p.shape[longest])) longest = int(d);
  if (longest >= 0) take(uint32_t(longest), p.shape[longest]);
  uint32_t n_act = n_first;
  fill_tile(t, p, ext, nullptr, nullptr, first, &n_act, blocks);
  t->tile = tile;
  for (uint32_t e = 0; e < 4; e++) t->lds_step[e] = 0;
  // In the destination's order, the second digit first: where that is 64 tiles and more of rows whole pages apart in the source, those under way read a narrow strip of
  // every row, a few memory channels.  Along the source's rows, each one tile further on, both sides spread (us, before / after: f32 2048 x 16384 into
  // bf16 strips of 16 41.9 / 39.8, 8192 x 8192 81.8 / 75.7, f32 to f32 120.2 / 100.1, bf16 4096 x 4096 15.2 / 12.5, 8192 x 128 x 32 turned to 128 x 8192 23.6 / 18.3).  Not for fewer
  // tiles (f32 strips of 16 back into 8192 x 8192, 16 of them, 95.0 / 103.4), other rows (strips back into 1000 x 80000 116.0 / 121.8), where the caches hold the
  // tensors (2000 x 3008 9.2 / 9.6), for runs of 16 bytes (bf16 4096 x 4096 strips of 8 15.3 / 15.9), or onto wider elements, where the writes are the larger part
  // (bf16 2048 x 16384 into f32 strips of 16 31.5 / 34.6).
  const int64_t apart = n_first > 1 ? p.ss[first[1]] * int64_t(vec * se) : 0;
  t->diagonal = se >= de && vec * se >= 16 && ext[shared] * vec * se >= 32 && t->chunks[1] >= 64 && apart >= 8192 && apart % 4096 == 0 &&
                p.count * vec * (se + de) >= 64000000;
  return *blocks < (1u << 24) ? tile : 0;
}

// k_move_runs: `shared` is the digit both sides store contiguously, in vectors of `vec` elements.
hipError_t launch_move_runs(MoveStrided p, uint32_t shared, uint32_t vec, bool tiled, hipStream_t stream) {
  const uint32_t se = uint32_t(mrl_dtype_size(p.sdt)), de = uint32_t(mrl_dtype_size(p.ddt));
  for (uint32_t d = 0; d < p.rank; d++) {
    if (d == shared) p.shape[d] /= vec;
    else p.ss[d] /= vec, p.ds[d] /= vec;
  }
  p.count /= vec;
  MoveTile t;
  uint64_t blocks = 0;
  // (a tile that leaves threads of its workgroup without a vector: four short digits, the rest of the tensor elsewhere)
  const uint32_t tile = tiled ? runs_tile(p, shared, vec, se, de, &t, &blocks) : 0;
  if (tile < 192) {
    blocks = (p.count + 255) / 256;
    for (uint32_t o = 0; o < p.rank; o++) p.by_shape[o] = FastDiv(p.shape[p.order[o]]);
  }
  const dim3 grid{uint32_t(blocks)};
#define MRL_RUNS_V(SE, DE, V)                                                                                       \
  if (vec == V) {                                                                                                  \
    if (tile < 192) MRL_LAUNCH((k_move_runs<SE, DE, V>), grid, dim3(256), 0, stream, p);                            \
    else if (tile > 256 && t.diagonal) {                                                                            \
      if constexpr (SE >= DE && V * SE >= 16) MRL_LAUNCH((k_move_runs<SE, DE, V, 4, true>), grid, dim3(256), 0, stream, t); \
    } else if (tile > 256) MRL_LAUNCH((k_move_runs<SE, DE, V, 4>), grid, dim3(256), 0, stream, t);                  \
    else MRL_LAUNCH((k_move_runs<SE, DE, V, 1>), grid, dim3(256), 0, stream, t);                                    \
  }
#define MRL_RUNS(SE, DE)                                                                                            \
  if (se == SE && de == DE) {                                                                                      \
    constexpr int WIDE = 16 / (SE > DE ? SE : DE);                                                                  \
    if constexpr (SE == 4 && DE == 2) MRL_RUNS_V(SE, DE, 8)                                                         \
    MRL_RUNS_V(SE, DE, WIDE)                                                                                        \
    else MRL_RUNS_V(SE, DE, WIDE / 2)                                                                               \
    else if constexpr (WIDE >= 8) MRL_RUNS_V(SE, DE, WIDE / 4)                                                      \
  }
  MRL_RUNS(1, 1) MRL_RUNS(1, 2) MRL_RUNS(1, 4)
  MRL_RUNS(2, 1) MRL_RUNS(2, 2) MRL_RUNS(2, 4)
  MRL_RUNS(4, 1) MRL_RUNS(4, 2) MRL_RUNS(4, 4)
#undef MRL_RUNS
#undef MRL_RUNS_V
  return mrl::plan::last_error();
}
}  // namespace

// Move over a common strided view of the two sides (layout_factor.h).  Returns
// hipErrorInvalidValue when the view does not fit the kernels' index ranges (the caller then
// takes the generic path).
hipError_t launch_move_view(const void *src, int src_dtype, void *dst, int dst_dtype,
                            const MoveDim *dims, uint32_t rank, hipStream_t stream) {
  if (rank > MOVE_MAX_RANK) return hipErrorInvalidValue;
  {
    double count = 1;
    for (uint32_t d = 0; d < rank; d++) count *= dims[d].size;
    plan::work(plan::UNIT_STREAM, 0, count * (mrl_dtype_size(src_dtype) + mrl_dtype_size(dst_dtype)));
  }
  // Elements narrower than 4 bytes that travel together (a digit contiguous on both sides, no
  // conversion) are moved as 2- or 4-byte units: a Packed(4) digit of bytes becomes one u32.
  MoveDim wide[MOVE_MAX_RANK];
  if (src_dtype == dst_dtype && mrl_dtype_size(src_dtype) < 4) {
    const uint32_t elem = uint32_t(mrl_dtype_size(src_dtype));
    for (uint32_t unit = 4; unit > elem; unit /= 2) {
      const uint32_t per = unit / elem;
      int shared = -1;
      bool fits = (reinterpret_cast<uintptr_t>(src) % unit) == 0 && (reinterpret_cast<uintptr_t>(dst) % unit) == 0;
      for (uint32_t d = 0; d < rank; d++)
        if (dims[d].size > 1 && dims[d].ss == 1 && dims[d].ds == 1) shared = int(d);
      for (uint32_t d = 0; fits && d < rank; d++)
        fits = int(d) == shared ? dims[d].size % per == 0 : (dims[d].ss % per == 0 && dims[d].ds % per == 0);
      if (shared < 0 || !fits) continue;
      uint32_t n = 0;
      for (uint32_t d = 0; d < rank; d++) {
        MoveDim m = dims[d];
        if (int(d) == shared) m.size /= per;
        else m.ss /= per, m.ds /= per;
        if (m.size > 1) wide[n++] = m;
      }
      if (n == 0) wide[n++] = {1, 1, 1};
      dims = wide, rank = n;
      src_dtype = dst_dtype = unit == 4 ? MRL_U32 : MRL_U16;
      break;
    }
  }
  MoveStrided p;
  p.src = src, p.dst = dst, p.sdt = src_dtype, p.ddt = dst_dtype, p.rank = rank;
  p.count = 1;
  int dim_s = -1, dim_d = -1;
  for (uint32_t d = 0; d < MOVE_MAX_RANK; d++) {
    p.shape[d] = d < rank ? dims[d].size : 1;
    p.ss[d] = d < rank ? dims[d].ss : 0;
    p.ds[d] = d < rank ? dims[d].ds : 0;
    p.count *= p.shape[d];
    if (d < rank && p.shape[d] > 1 && p.ss[d] == 1) dim_s = int(d);
    if (d < rank && p.shape[d] > 1 && p.ds[d] == 1) dim_d = int(d);
  }
  if (p.count == 0) return hipSuccess;
  if (p.count > 0xffffffffull) return hipErrorInvalidValue;  // the kernels index elements with 32 bits
  // Decode order: by decreasing destination stride, the destination's contiguous dim last.
  for (uint32_t d = 0; d < MOVE_MAX_RANK; d++) p.order[d] = d;
  for (uint32_t i = 0; i < p.rank; i++)
    for (uint32_t j = i + 1; j < p.rank; j++)
      if (p.ds[p.order[j]] > p.ds[p.order[i]]) std::swap(p.order[i], p.order[j]);
  const size_t se = mrl_dtype_size(src_dtype), de = mrl_dtype_size(dst_dtype);
  const bool shared = dim_s >= 0 && dim_s == dim_d;
  if (shared && rank == 1) {
    if (src_dtype == dst_dtype && p.count % (16 / se) == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0 &&
        (reinterpret_cast<uintptr_t>(dst) & 15) == 0)
      return launch_copy(src, dst, p.count * se, stream);
    // One contiguous run with a conversion: four elements per thread.
    if (src_dtype != dst_dtype && p.count >= 1024 &&
        (reinterpret_cast<uintptr_t>(src) % (4 * se)) == 0 && (reinterpret_cast<uintptr_t>(dst) % (4 * de)) == 0) {
      // sixteen bytes a thread on the wider side where both buffers are aligned for it
      // (two-byte to one-byte elements: sixteen, two 16-byte loads and a 16-byte store)
      const uint32_t wide = se == 2 && de == 1 ? 16u : uint32_t(16 / std::max(se, de));
      const uint32_t n = (reinterpret_cast<uintptr_t>(src) % (wide * se)) == 0 && (reinterpret_cast<uintptr_t>(dst) % (wide * de)) == 0 ? wide : 4;
      const uint32_t blocks = uint32_t(std::min<uint64_t>((p.count / n + 255) / 256, 1u << 20));
      const dim3 grid{blocks}, block{256};
#define MRL_CONVERT(SE, DE)                                                                                                  \
  if (se == SE && de == DE) {                                                                                                \
    constexpr int WIDE = SE == 2 && DE == 1 ? 16 : 16 / (SE > DE ? SE : DE);                                                 \
    if (n == WIDE) MRL_LAUNCH((k_convert4<SE, DE, WIDE>), grid, block, 0, stream, src, dst, src_dtype, dst_dtype, p.count);   \
    else MRL_LAUNCH((k_convert4<SE, DE, 4>), grid, block, 0, stream, src, dst, src_dtype, dst_dtype, p.count);               \
  }
      MRL_CONVERT(1, 1) MRL_CONVERT(1, 2) MRL_CONVERT(1, 4)
      MRL_CONVERT(2, 1) MRL_CONVERT(2, 2) MRL_CONVERT(2, 4)
      MRL_CONVERT(4, 1) MRL_CONVERT(4, 2) MRL_CONVERT(4, 4)
#undef MRL_CONVERT
      return mrl::plan::last_error();
    }
  }
  // A shared contiguous digit in whole vectors on both sides: 16, 8 or 4 bytes on the wider side.
  // From 32-bit elements to 16-bit ones 16 bytes on the narrower side where the source's rows lie 8, 16, 32 or 64 KiB apart, on the
  // same memory channels (us, four elements a vector / eight: f32 2048 x 16384 into bf16 strips of 16 44.9 / 42.2, 4096 x 16384 109 / 84, 8192 x 8192 98 / 82, 1024 x 4096 8.7 /
  // 7.9, 2048 x 2048 9.0 / 8.0; other rows: 2048 x 12288 30.3 / 33.3, 2048 x 10240 25.3 / 28.0, 8192 x 6144 58.6 / 62.1, 1024 x 32768 39.7 / 41.6).
  const size_t widest = std::max(se, de);
  uint32_t vec = 0;
  // `row`: bytes from one row of the source to the next, the source's step along the digit that continues the destination's runs:
  // the one that a tile is long along.  (The longest stride of a batched Move is the entries': 2 x 8192 x 3072 63.7 us with eight
  // elements a vector, 61.4 with four, 8 x 1024 x 1536 18.5 and 16.4.)
  uint64_t row = 0;
  int64_t least = 0;
  for (uint32_t d = 0; d < rank; d++)
    if (int(d) != dim_d && p.shape[d] > 1 && (row == 0 || p.ds[d] < least)) row = uint64_t(p.ss[d]) * se, least = p.ds[d];
  const bool pages = se == 4 && de == 2 && p.count > MOVE_SMALL && (row == 8192 || row == 16384 || row == 32768 || row == 65536);
  if (shared && rank > 1)
    for (uint32_t v = uint32_t(16 / widest) * (pages ? 2 : 1); vec == 0 && v >= 1 && v * widest >= 4; v /= 2) {
      bool fits = v > 1 && p.shape[dim_s] % v == 0 && (reinterpret_cast<uintptr_t>(src) % std::min<size_t>(16, v * se)) == 0 &&
                  (reinterpret_cast<uintptr_t>(dst) % (v * de)) == 0;
      for (uint32_t d = 0; fits && d < rank; d++) fits = int(d) == dim_s || (p.ss[d] % v == 0 && p.ds[d] % v == 0);
      if (fits) vec = v;
    }
  const bool small = p.count <= MOVE_SMALL;
  if (vec) {
    const bool long_runs = vec == 16 / widest && se == de && uint64_t(p.shape[dim_s]) * se >= 64 && p.count * se <= MOVE_DIRECT_BYTES;
    return launch_move_runs(p, uint32_t(dim_s), vec, !small && !long_runs, stream);
  }
  // Runs of at least 64 bytes that are not whole vectors (odd rows), a tensor of one round of
  // workgroups either way, or one with no contiguous digit: an element per thread.
  const bool shared_runs = shared && (rank == 1 || uint64_t(p.shape[dim_s]) * se >= 64);
  const bool tiny = p.count <= MOVE_TINY;
  if (dim_s < 0 || dim_d < 0 || shared_runs || tiny) {
    const uint64_t blocks = (p.count + 255) / 256;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    for (uint32_t o = 0; o < rank; o++) p.by_shape[o] = FastDiv(p.shape[p.order[o]]);
    MRL_LAUNCH(k_move_rows, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    return mrl::plan::last_error();
  }
  // Two long contiguous dims: the 64 x 64 transpose.
  if (dim_s != dim_d && p.shape[dim_s] >= 32 && p.shape[dim_d] >= 32) {
    p.dim_s = uint32_t(dim_s), p.dim_d = uint32_t(dim_d);
    // 16-bit elements, nothing converted, every dword whole and aligned: two elements per lane.
    bool pairs = src_dtype == dst_dtype && mrl_dtype_size(src_dtype) == 2 && p.shape[dim_s] % 2 == 0 &&
                 p.shape[dim_d] % 2 == 0 && (reinterpret_cast<uintptr_t>(src) & 3) == 0 &&
                 (reinterpret_cast<uintptr_t>(dst) & 3) == 0;
    for (uint32_t d = 0; pairs && d < p.rank; d++)
      pairs = (int(d) == dim_s || p.ss[d] % 2 == 0) && (int(d) == dim_d || p.ds[d] % 2 == 0);
    // ... and the source side in whole 16-byte vectors.
    bool octets = pairs && p.shape[dim_s] % 8 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0;
    for (uint32_t d = 0; octets && d < p.rank; d++) octets = int(d) == dim_s || p.ss[d] % 8 == 0;
    // Bytes: sixteen per lane on the source side, four on the destination side.
    bool bytes16 = src_dtype == dst_dtype && mrl_dtype_size(src_dtype) == 1 && p.shape[dim_s] % 16 == 0 &&
                   p.shape[dim_d] % 4 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(dst) & 3) == 0;
    for (uint32_t d = 0; bytes16 && d < p.rank; d++)
      bytes16 = (int(d) == dim_s || p.ss[d] % 16 == 0) && (int(d) == dim_d || p.ds[d] % 4 == 0);
    // 32-bit elements likewise, four per lane.
    bool quads = src_dtype == dst_dtype && mrl_dtype_size(src_dtype) == 4 && p.shape[dim_s] % 4 == 0 &&
                 p.shape[dim_d] % 4 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0 &&
                 (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
    for (uint32_t d = 0; quads && d < p.rank; d++)
      quads = (int(d) == dim_s || p.ss[d] % 4 == 0) && (int(d) == dim_d || p.ds[d] % 4 == 0);
    const uint32_t side = pairs || bytes16 ? 128 : 64;
    p.tiles_s = (p.shape[dim_s] + side - 1) / side, p.tiles_d = (p.shape[dim_d] + side - 1) / side;
    uint64_t blocks = uint64_t(p.tiles_s) * p.tiles_d;
    for (uint32_t d = 0; d < p.rank; d++)
      if (int(d) != dim_s && int(d) != dim_d) blocks *= p.shape[d];
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    if (bytes16) MRL_LAUNCH(k_move_tiled8v, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    else if (octets) MRL_LAUNCH(k_move_tiled16v, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    else if (pairs) MRL_LAUNCH(k_move_tiled16, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    else if (quads) MRL_LAUNCH(k_move_tiled32, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    else if (src_dtype != dst_dtype) {
      const int se = int(mrl_dtype_size(src_dtype)), de = int(mrl_dtype_size(dst_dtype));
#define MRL_TILED(SE, DE) \
  if (se == SE && de == DE) MRL_LAUNCH((k_move_tiled<SE, DE>), dim3(uint32_t(blocks)), dim3(256), 0, stream, p)
      MRL_TILED(1, 1); MRL_TILED(1, 2); MRL_TILED(1, 4);
      MRL_TILED(2, 1); MRL_TILED(2, 2); MRL_TILED(2, 4);
      MRL_TILED(4, 1); MRL_TILED(4, 2); MRL_TILED(4, 4);
#undef MRL_TILED
    }
    else if (mrl_dtype_size(src_dtype) == 1) MRL_LAUNCH(k_move_tiled_as<uint8_t>, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    else if (mrl_dtype_size(src_dtype) == 2) MRL_LAUNCH(k_move_tiled_as<uint16_t>, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    else MRL_LAUNCH(k_move_tiled_as<uint32_t>, dim3(uint32_t(blocks)), dim3(256), 0, stream, p);
    return mrl::plan::last_error();
  }
  if (small) {
    const dim3 grid{uint32_t((p.count + 255) / 256)};
    for (uint32_t o = 0; o < rank; o++) p.by_shape[o] = FastDiv(p.shape[p.order[o]]);
#define MRL_GATHER(SE, DE) if (se == SE && de == DE) MRL_LAUNCH((k_move_gather<SE, DE>), grid, dim3(256), 0, stream, p);
    MRL_GATHER(1, 1) MRL_GATHER(1, 2) MRL_GATHER(1, 4)
    MRL_GATHER(2, 1) MRL_GATHER(2, 2) MRL_GATHER(2, 4)
    MRL_GATHER(4, 1) MRL_GATHER(4, 2) MRL_GATHER(4, 4)
#undef MRL_GATHER
    return mrl::plan::last_error();
  }
  // Otherwise a tile grown digit by digit: along the destination's fastest digits until they
  // make a run of 64, along the source's fastest until they do, then along the destination's
  // again while the tile stays within `cap`: 4096 elements, fewer where that would leave compute
  // units without a workgroup.
  const uint32_t cap = p.count >= 4096ull * 2 * g_compute_units ? MOVE_TILE_MAX : 1024;
  uint32_t ext[MOVE_MAX_RANK];
  uint32_t by_ss[MOVE_MAX_RANK], by_ds[MOVE_MAX_RANK];  // digits, fastest first
  for (uint32_t d = 0; d < MOVE_MAX_RANK; d++) by_ss[d] = by_ds[d] = d, ext[d] = 1;
  std::sort(by_ss, by_ss + rank, [&](uint32_t x, uint32_t y) { return p.ss[x] < p.ss[y]; });
  std::sort(by_ds, by_ds + rank, [&](uint32_t x, uint32_t y) { return p.ds[x] < p.ds[y]; });
  uint32_t tile = 1;
  auto grow = [&](const uint32_t *order, uint32_t run_target, uint32_t tile_cap) {
    uint32_t run = 1;
    for (uint32_t i = 0; i < rank && run < run_target; i++) {
      const uint32_t d = order[i];
      run *= ext[d];
      if (ext[d] == p.shape[d] || run >= run_target) continue;
      const uint32_t want = std::min<uint32_t>({p.shape[d] / ext[d], (run_target + run - 1) / run,
                                                std::max<uint32_t>(1, tile_cap / tile)});
      if (want <= 1) break;
      tile = tile / ext[d] * (ext[d] * want), run *= want, ext[d] *= want;
      if (ext[d] != p.shape[d]) break;  // a partly covered digit ends the contiguous run
    }
  };
  grow(by_ds, 64, cap / 64);
  grow(by_ss, 64, cap);
  grow(by_ds, cap, cap);
  // The runs are as long as they get; a tile still far below the cap (a digit covered in part
  // ends the growth above: 4 of 6 strips of an OddEven(16) dim left a tile of 64 elements, 20000
  // workgroups for 5 MB) is filled along whatever digits have room, more runs per workgroup.
  for (uint32_t i = 0; i < rank && tile < cap; i++) {
    const uint32_t d = by_ds[i];
    const uint32_t grown = std::min<uint32_t>(p.shape[d], uint32_t(uint64_t(ext[d]) * (cap / tile)));
    if (grown > ext[d]) tile = tile / ext[d] * grown, ext[d] = grown;
  }
  if (tile > MOVE_TILE_MAX) return hipErrorInvalidValue;
  uint32_t tstride_s[MOVE_MAX_RANK], tstride_d[MOVE_MAX_RANK];
  {
    uint32_t run_s = 1, run_d = 1;
    for (uint32_t d = 0; d < MOVE_MAX_RANK; d++) tstride_s[d] = tstride_d[d] = 1;
    for (uint32_t i = 0; i < rank; i++) {
      tstride_s[by_ss[i]] = run_s, run_s *= ext[by_ss[i]];
      tstride_d[by_ds[i]] = run_d, run_d *= ext[by_ds[i]];
    }
  }
  // Whether the tile's elements, taken in one side's order, lie there in whole runs of v (4 or 2): the
  // fastest digits continue each other (1, ext, ...) up to a multiple of v, inside the tensor as
  // well as inside the tile, and everything else is a multiple of v apart.  in_run: how many
  // of the fastest digits make up the run; on the destination side, whose runs are gathered from
  // LDS at fixed distances, no run may carry into a further digit.
  auto runs_of = [&](uint32_t v, const uint32_t *order, const int64_t *stride, const void *base, size_t size, bool gathered, uint32_t *in_run) {
    if ((reinterpret_cast<uintptr_t>(base) % (v * size)) != 0) return false;
    int64_t run = 1;
    for (uint32_t i = 0; i < rank; i++) {
      const uint32_t d = order[i];
      if (stride[d] != run || (gathered && v % run != 0)) return false;
      const bool whole = (run * ext[d]) % v == 0 && (run * p.shape[d]) % v == 0;
      if (whole) {
        for (uint32_t j = i + 1; j < rank; j++)
          if (stride[order[j]] % v != 0) return false;
        *in_run = i + 1;
        return true;
      }
      if (ext[d] != p.shape[d]) return false;
      run *= ext[d];
    }
    return false;
  };
  uint32_t digits_s = 0, digits_d = 0, run_s = 1, run_d = 1;
  for (uint32_t v : {4u, 2u}) {   // (two bytes are no wider than one)
    if (run_s == 1 && v * se >= 4 && runs_of(v, by_ss, p.ss, src, se, false, &digits_s)) run_s = v;
    if (run_d == 1 && v * de >= 4 && runs_of(v, by_ds, p.ds, dst, de, true, &digits_d)) run_d = v;
  }
  MoveTile t;
  for (uint32_t e = 0; e < 4; e++) {
    uint32_t rem = e;
    t.lds_step[e] = 0;
    for (uint32_t i = 0; run_d > 1 && i < digits_d; i++) {
      const uint32_t d = by_ds[i], size = i + 1 == digits_d ? run_d : ext[d];
      t.lds_step[e] += rem % size * tstride_s[d], rem /= size;
    }
  }
  uint32_t n_act = 0;
  uint64_t blocks = 0;
  fill_tile(&t, p, ext, tstride_s, tstride_d, nullptr, &n_act, &blocks);
  t.tile = tile;
  if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
  if (se == 1) return launch_move_gather<1>(t, uint32_t(de), run_s, run_d, n_act, uint32_t(blocks), stream);
  if (se == 2) return launch_move_gather<2>(t, uint32_t(de), run_s, run_d, n_act, uint32_t(blocks), stream);
  return launch_move_gather<4>(t, uint32_t(de), run_s, run_d, n_act, uint32_t(blocks), stream);
}

// Move between two strided layouts of the same logical shape.
hipError_t launch_move_strided(const Strided &src, const Strided &dst, hipStream_t stream) {
  // Dims of size one address nothing; neighbours that continue each other on both sides (h and w
  // of an image between NCHW and NHWC) are one dim: the tiled kernels then see its whole length
  // (56 x 56 pixels as 3136, whole 16-byte vectors, where a row of 56 is not).
  MoveDim dims[MRL_MAX_RANK];
  uint32_t n = 0;
  for (uint32_t d = 0; d < src.rank; d++) {
    if (src.shape[d] == 1) continue;
    const MoveDim next = {src.shape[d], src.stride[d], dst.stride[d]};
    if (n > 0 && dims[n - 1].ss == next.ss * int64_t(next.size) && dims[n - 1].ds == next.ds * int64_t(next.size) &&
        uint64_t(dims[n - 1].size) * next.size <= 0xffffffffull)
      dims[n - 1] = {dims[n - 1].size * next.size, next.ss, next.ds};
    else
      dims[n++] = next;
  }
  if (n == 0) dims[n++] = {1, 1, 1};
  return launch_move_view(src.ptr, src.dtype, dst.ptr, dst.dtype, dims, n, stream);
}

bool pad_rows_possible(const PadRows &p) {
  const Strided &src = p.src;
  if (src.rank != 3 || (src.shape[2] != 1 && src.stride[2] != 1) || uint64_t(p.dst_ld) * p.elem_size % 16 != 0 || p.dst_ld < src.shape[2] ||
      p.dst_rows < src.shape[1])
    return false;
  const double chunks = double(src.shape[0]) * p.dst_rows * (uint64_t(p.dst_ld) * p.elem_size / 16);
  return chunks >= 1 && chunks < double(1u << 31);
}

namespace {
bool pad_job(const PadRows &p, PadJob *j) {
  if (!pad_rows_possible(p) || (reinterpret_cast<uintptr_t>(p.dst) & 15) != 0) return false;
  const Strided &src = p.src;
  const uint32_t es = p.elem_size, batch = src.shape[0], rows = src.shape[1];
  j->src = static_cast<const uint8_t *>(src.ptr), j->dst = static_cast<chunk_t *>(p.dst);
  j->rows = rows, j->dst_rows = p.dst_rows, j->row_bytes = uint64_t(src.shape[2]) * es, j->row_chunks = uint32_t(uint64_t(p.dst_ld) * es / 16);
  j->chunks = batch * p.dst_rows * j->row_chunks;
  j->src_batch = (batch == 1 ? 0 : src.stride[0]) * int64_t(es), j->src_ld = (rows == 1 ? 0 : src.stride[1]) * int64_t(es);
  j->by_row_chunks = FastDiv(j->row_chunks), j->by_dst_rows = FastDiv(j->dst_rows);
  j->panel_chunks = p.panel * es / 16, j->by_panel_chunks = FastDiv(std::max(1u, j->panel_chunks));
  return true;
}
// Four chunks a thread, their loads in flight together, for copies that fill the chip several times over; below, one a
// thread, a shorter way to the first load (whole Matmuls of random sizes, four / one, geometric means by chunks of the larger
// operand: 16 thousand 8.1 / 7.3 us, 256 thousand 20.6 / 19.8, 1 Mi 37.4 / 37.2, 4 Mi 97.0 / 100.6).
bool pad_in_fours(uint32_t chunks) { return chunks >= 4096ull * g_compute_units; }
double pad_bytes(const PadJob &j) { return double(j.chunks) / j.row_chunks / j.dst_rows * j.rows * j.row_bytes + 16.0 * j.chunks; }
}  // namespace

hipError_t launch_pad_rows(const PadRows &p, hipStream_t stream) {
  PadJob j;
  if (!pad_job(p, &j)) return hipErrorInvalidValue;
  plan::work(plan::UNIT_STREAM, 0, pad_bytes(j));
  if (pad_in_fours(j.chunks)) MRL_LAUNCH((k_pad_rows<PAD_UNROLL>), dim3((j.chunks + 256 * PAD_UNROLL - 1) / (256 * PAD_UNROLL)), dim3(256), 0, stream, j);
  else MRL_LAUNCH((k_pad_rows<1>), dim3((j.chunks + 255) / 256), dim3(256), 0, stream, j);
  return mrl::plan::last_error();
}

hipError_t launch_pad_rows_pair(const PadRows &p0, const PadRows &p1, hipStream_t stream) {
  PadJob j0, j1;
  if (!pad_job(p0, &j0) || !pad_job(p1, &j1)) return hipErrorInvalidValue;
  // The larger first: workgroups of the smaller that have nothing to copy then stand at the launch's end (bf16 1344 x 1111 x 5021 33.7 / 33.0 us).
  if (j0.chunks < j1.chunks) std::swap(j0, j1);
  plan::work(plan::UNIT_STREAM, 0, pad_bytes(j0) + pad_bytes(j1));
  const uint32_t most = std::max(j0.chunks, j1.chunks);
  if (pad_in_fours(most)) MRL_LAUNCH((k_pad_rows_pair<PAD_UNROLL>), dim3((most + 256 * PAD_UNROLL - 1) / (256 * PAD_UNROLL), 2), dim3(256), 0, stream, j0, j1);
  else MRL_LAUNCH((k_pad_rows_pair<1>), dim3((most + 255) / 256, 2), dim3(256), 0, stream, j0, j1);
  return mrl::plan::last_error();
}

hipError_t launch_widen_bf16(const void *src, void *dst, uint64_t count, hipStream_t stream) {
  if (count == 0) return hipSuccess;
  uint64_t blocks = (count + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  plan::work(plan::UNIT_STREAM, 0, 6.0 * count);
  MRL_LAUNCH(k_widen_bf16, dim3(uint32_t(blocks)), dim3(256), 0, stream, (const uint16_t *)src,
                     (uint32_t *)dst, count);
  return mrl::plan::last_error();
}

hipError_t launch_matmul_generic(const Strided &a, const Strided &b, const Strided &c, int accum,
                                 hipStream_t stream) {
  MM p;
  p.a = a.ptr, p.b = b.ptr, p.c = c.ptr;
  p.dta = a.dtype, p.dtb = b.dtype, p.dtc = c.dtype;
  p.B = a.shape[0], p.M = a.shape[1], p.K = a.shape[2], p.N = b.shape[2];
  for (int d = 0; d < 3; d++) p.sa[d] = a.stride[d], p.sb[d] = b.stride[d], p.sc[d] = c.stride[d];
  p.accum = accum;
  const uint64_t tiles = uint64_t((p.N + 15) / 16) * ((p.M + 15) / 16) * p.B;
  if (tiles > 0x7fffffffull) return hipErrorInvalidValue;
  dim3 grid{uint32_t(tiles)};
  {
    const double mn = double(p.B) * p.M * p.N;
    plan::work(plan::UNIT_VALU, 2.0 * mn * p.K,
               double(p.B) * (double(p.M) * p.K * mrl_dtype_size(a.dtype) + double(p.K) * p.N * mrl_dtype_size(b.dtype)) +
                   mn * mrl_dtype_size(c.dtype));
  }
  if (float_out(c.dtype)) MRL_LAUNCH(k_matmul_generic<true>, grid, dim3(256), 0, stream, p);
  else MRL_LAUNCH(k_matmul_generic<false>, grid, dim3(256), 0, stream, p);
  return mrl::plan::last_error();
}

hipError_t launch_conv_generic(const Strided &img, const Strided &filt, const Strided &out,
                               int accum, hipStream_t stream) {
  CV p;
  p.img = img.ptr, p.filt = filt.ptr, p.out = out.ptr;
  p.dti = img.dtype, p.dtf = filt.dtype, p.dto = out.dtype;
  p.B = out.shape[0], p.F = out.shape[1], p.OH = out.shape[2], p.OW = out.shape[3];
  p.C = filt.shape[1], p.FH = filt.shape[2], p.FW = filt.shape[3];
  for (int d = 0; d < 4; d++) p.si[d] = img.stride[d], p.sf[d] = filt.stride[d], p.so[d] = out.stride[d];
  p.accum = accum;
  const uint64_t total = uint64_t(p.B) * p.F * p.OH * p.OW;
  plan::work(plan::UNIT_VALU, 2.0 * total * p.C * p.FH * p.FW,
             double(p.B) * p.C * (p.OH + p.FH - 1) * (p.OW + p.FW - 1) * mrl_dtype_size(img.dtype) +
                 double(total) * mrl_dtype_size(out.dtype));
  if (total <= 16384 && uint64_t(p.C) * p.FH * p.FW >= 32) {  // few outputs, long reductions
    const uint32_t wave_blocks = uint32_t((total + 3) / 4);
    if (float_out(out.dtype)) MRL_LAUNCH(k_conv_generic_wave<true>, dim3(wave_blocks), dim3(256), 0, stream, p);
    else MRL_LAUNCH(k_conv_generic_wave<false>, dim3(wave_blocks), dim3(256), 0, stream, p);
    return mrl::plan::last_error();
  }
  const uint32_t blocks = uint32_t((total + 255) / 256);
  if (float_out(out.dtype)) MRL_LAUNCH(k_conv_generic<true>, dim3(blocks), dim3(256), 0, stream, p);
  else MRL_LAUNCH(k_conv_generic<false>, dim3(blocks), dim3(256), 0, stream, p);
  return mrl::plan::last_error();
}

// Pieces the scan dim is cut into when the column kernel would have `blocks` workgroups: none
// (1) when those fill the chip or the scan dim is short; else enough for about 1024 workgroups,
// each piece at least 32 steps (a 256-thread workgroup takes 32 steps in one unrolled pass).
uint32_t softmax_cols_chunks(uint64_t blocks, uint32_t scan) {
  if (blocks >= 256 || scan < 128) return 1;
  const uint64_t want = (1024 + blocks - 1) / blocks;
  return uint32_t(std::max<uint64_t>(1, std::min<uint64_t>({want, scan / 32, 256})));
}

size_t softmax_cols_scratch_bytes(uint64_t blocks, uint32_t scan) {
  const uint32_t chunks = softmax_cols_chunks(blocks, scan);
  return chunks > 1 ? size_t(blocks) * chunks * 64 * sizeof(float2) : 0;
}

hipError_t launch_softmax_generic(const Strided &in, const Strided &out, uint32_t scan_dim, void *scratch,
                                  hipStream_t stream) {
  SM p;
  p.in = (const float *)in.ptr, p.out = (float *)out.ptr;
  p.rank = in.rank, p.scan_dim = scan_dim;
  uint64_t lines = 1;
  for (uint32_t d = 0; d < MRL_MAX_RANK; d++) {
    p.shape[d] = d < in.rank ? in.shape[d] : 1;
    p.si[d] = d < in.rank ? in.stride[d] : 0;
    p.so[d] = d < in.rank ? out.stride[d] : 0;
    if (d < in.rank && d != scan_dim) lines *= in.shape[d];
  }
  p.lines = lines;
  plan::work(plan::UNIT_VALU, 20.0 * lines * in.shape[scan_dim], 8.0 * lines * in.shape[scan_dim]);
  // A dim other than the scan dim that both sides store contiguously: the column kernel.
  for (uint32_t d = 0; d < in.rank; d++)
    if (d != scan_dim && in.shape[d] >= 16 && in.stride[d] == 1 && out.stride[d] == 1) {
      SMC q;
      q.s = p, q.fast = d, q.fast_tiles = (in.shape[d] + 63) / 64;
      q.chunks = 1, q.chunk_len = in.shape[scan_dim], q.pairs = nullptr;
      if (in.shape[scan_dim] <= 16 && lines >= 65536) {
        q.fast_tiles = (in.shape[d] + 255) / 256;
        const uint64_t wgs = lines / in.shape[d] * q.fast_tiles;
        if (wgs > 0x7fffffffull) break;
        MRL_LAUNCH(k_softmax_cols_short, dim3(uint32_t(wgs)), dim3(256), 0, stream, q);
        return mrl::plan::last_error();
      }
      const uint64_t blocks = lines / in.shape[d] * q.fast_tiles;
      if (blocks > 0x7fffffffull) break;
      const uint32_t chunks = scratch ? softmax_cols_chunks(blocks, in.shape[scan_dim]) : 1;
      const bool runs = in.stride[scan_dim] % 32 != 0 || out.stride[scan_dim] % 32 != 0;
      if (chunks > 1) {
        // Few columns: the scan dim shared out over blockIdx.y as well, in two launches.
        q.chunks = chunks, q.chunk_len = (in.shape[scan_dim] + chunks - 1) / chunks, q.pairs = (float2 *)scratch;
        const double count = double(lines) * in.shape[scan_dim];
        // Measured 2.5-4.4 TB/s over their 12 bytes an element; a workgroup's chain of passes over
        // its piece (32 steps a pass) is what small problems take: 2149 x 172 11 us, 100000 x 64 45 us.
        const double chain_ns = 2500.0 + 700.0 * ((q.chunk_len + 31) / 32);
        plan::work(plan::UNIT_STREAM, 0, 5.2 * count, 0, chain_ns);
        if (runs) MRL_LAUNCH((k_softmax_cols<4, 1, 0, true>), dim3(uint32_t(blocks), chunks), dim3(256), 0, stream, q);
        else MRL_LAUNCH((k_softmax_cols<4, 1>), dim3(uint32_t(blocks), chunks), dim3(256), 0, stream, q);
        plan::work(plan::UNIT_STREAM, 0, 10.4 * count, 0, chain_ns);
        if (runs) MRL_LAUNCH((k_softmax_cols<4, 2, 0, true>), dim3(uint32_t(blocks), chunks), dim3(256), 0, stream, q);
        else MRL_LAUNCH((k_softmax_cols<4, 2>), dim3(uint32_t(blocks), chunks), dim3(256), 0, stream, q);
        return mrl::plan::last_error();
      }
      // Columns in registers while two workgroups of sixteen waves share a compute unit with them (32 values a lane); with 64 values
      // 32 x 541 x 587 took 49.0 us against 36.2 read twice.
      const uint32_t scan = in.shape[scan_dim];
      const dim3 grid(uint32_t(blocks), 1, 1);
      if (scan <= 64) MRL_LAUNCH((k_softmax_cols<4, 0, 16>), grid, dim3(256), 0, stream, q);
      else if (scan <= 128) MRL_LAUNCH((k_softmax_cols<4, 0, 32>), grid, dim3(256), 0, stream, q);
      else if (scan <= 256) MRL_LAUNCH((k_softmax_cols<8, 0, 32>), grid, dim3(512), 0, stream, q);
      else if (scan <= 512) MRL_LAUNCH((k_softmax_cols<16, 0, 32>), grid, dim3(1024), 0, stream, q);
      else if (runs) MRL_LAUNCH((k_softmax_cols<16, 0, 0, true>), grid, dim3(1024), 0, stream, q);
      else MRL_LAUNCH((k_softmax_cols<16, 0>), grid, dim3(1024), 0, stream, q);
      return mrl::plan::last_error();
    }
  const uint32_t blocks = uint32_t((lines + 3) / 4);
  MRL_LAUNCH(k_softmax_generic, dim3(blocks), dim3(256), 0, stream, p);
  return mrl::plan::last_error();
}

namespace {
// One thread per 32-bit element of C.
template <class T, class Stored = T>
__global__ __launch_bounds__(256) void k_sum_splits(const T *__restrict__ partial, Stored *__restrict__ c, uint32_t splits,
                                                    uint32_t n, uint64_t count, int64_t ldc, int accum) {
  const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= count) return;
  Stored *to = c + int64_t(i / n) * ldc + int64_t(i % n);
  T sum = accum ? T(*to) : T(0);
  constexpr uint32_t U = 8;  // loads in flight together
  for (uint32_t s0 = 0; s0 < splits; s0 += U) {
    T v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) v[u] = partial[uint64_t(s0 + u < splits ? s0 + u : s0) * count + i];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) sum += s0 + u < splits ? v[u] : T(0);
  }
  *to = Stored(sum);
}
}  // namespace

hipError_t launch_sum_splits(const void *partial, void *c, uint32_t splits, uint32_t m, uint32_t n, int64_t ldc,
                             bool accum, bool integers, bool c_bf16, hipStream_t stream) {
  const uint64_t count = uint64_t(m) * n;
  if (count == 0) return hipSuccess;
  const uint64_t blocks = (count + 255) / 256;
  if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
  plan::work(plan::UNIT_STREAM, 0, 4.0 * count * (splits + 1 + (accum ? 1 : 0)));
  if (integers)
    MRL_LAUNCH(k_sum_splits<int>, dim3(uint32_t(blocks)), dim3(256), 0, stream, (const int *)partial, (int *)c, splits, n,
               count, ldc, int(accum));
  else if (c_bf16)
    MRL_LAUNCH((k_sum_splits<float, __bf16>), dim3(uint32_t(blocks)), dim3(256), 0, stream, (const float *)partial, (__bf16 *)c, splits,
               n, count, ldc, int(accum));
  else
    MRL_LAUNCH(k_sum_splits<float>, dim3(uint32_t(blocks)), dim3(256), 0, stream, (const float *)partial, (float *)c, splits,
               n, count, ldc, int(accum));
  return mrl::plan::last_error();
}

hipError_t launch_fill_zero(void *ptr, uint64_t bytes, hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  const uint64_t words = bytes / 4;
  const uint32_t tail = uint32_t(bytes % 4);
  uint64_t blocks = (words + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks == 0) blocks = 1;
  plan::work(plan::UNIT_STREAM, 0, double(bytes));
  MRL_LAUNCH(k_fill_zero, dim3(uint32_t(blocks)), dim3(256), 0, stream, (uint32_t *)ptr,
                     words, (uint8_t *)ptr + words * 4, tail);
  return mrl::plan::last_error();
}

}  // namespace mrl
