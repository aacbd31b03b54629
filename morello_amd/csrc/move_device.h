// What the Move kernels share: elements of any dtype as bits, their conversions (Rust `as`), and a tile of a Move over a
// common strided view.
#pragma once
#include <type_traits>

#include "kernels.h"
#include "layout_factor.h"

namespace mrl {

// A tile of a Move over a common strided view: `ext[d]` elements along each digit, as many tiles along
// it as `chunks[d]`.  Element t of the tile in source order has digit (t / tstride_s[d]) % ext[d]
// along d, likewise tstride_d in destination order; the divisions are multiplications by
// precomputed reciprocals (exact for operands below 2^16).  The digits the tile extends along come
// first.
struct MoveTile {
  const void *src;
  void *dst;
  int sdt, ddt;
  uint32_t shape[MOVE_MAX_RANK];
  int64_t ss[MOVE_MAX_RANK], ds[MOVE_MAX_RANK];
  uint32_t ext[MOVE_MAX_RANK], chunks[MOVE_MAX_RANK];
  uint32_t tstride_s[MOVE_MAX_RANK], tstride_d[MOVE_MAX_RANK];
  uint32_t inv_s[MOVE_MAX_RANK], inv_d[MOVE_MAX_RANK], inv_ext[MOVE_MAX_RANK];  // ceil(2^32 / x)
  uint32_t tile;  // elements (k_move_runs: vectors) per tile
  FastDiv by_chunks[MOVE_MAX_RANK];   // a block number into tile coordinates without dividing (blocks number below 2^31)
  bool diagonal;         // k_move_runs: which of tile_origin's orders
  uint32_t lds_step[4];  // k_move_gather: where the elements of a destination run of four lie in source order, from its first
};
constexpr uint32_t MOVE_TILE_MAX = 4096;

// k_move_gather's launch (move_gather.h) for sources of SE bytes an element, in a translation unit for each.  run_s, run_d: elements
// per access on the two sides (4, 2 or 1); n_act: digits that the tile extends along.
template <int SE>
hipError_t launch_move_gather(const MoveTile &t, uint32_t dst_bytes, uint32_t run_s, uint32_t run_d, uint32_t n_act, uint32_t blocks, hipStream_t stream);
extern template hipError_t launch_move_gather<1>(const MoveTile &, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
extern template hipError_t launch_move_gather<2>(const MoveTile &, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);
extern template hipError_t launch_move_gather<4>(const MoveTile &, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, hipStream_t);

namespace {

__device__ inline float bf16_bits_to_f32(uint16_t v) { return __uint_as_float(uint32_t(v) << 16); }

__device__ inline uint32_t narrow_int(int dtype, uint32_t v) {
  switch (dtype) {
    case MRL_U8: return v & 0xffu;
    case MRL_I8: return uint32_t(int32_t(int8_t(uint8_t(v))));
    case MRL_U16: return v & 0xffffu;
    case MRL_I16: return uint32_t(int32_t(int16_t(uint16_t(v))));
    default: return v;
  }
}

// Rust `as` for narrow integer targets saturates floats at the target's own bounds.
__device__ inline uint32_t float_to_int(float f, int dt) {
  if (f != f) return 0;
  float lo, hi;
  switch (dt) {
    case MRL_U8: lo = 0.f, hi = 255.f; break;
    case MRL_I8: lo = -128.f, hi = 127.f; break;
    case MRL_U16: lo = 0.f, hi = 65535.f; break;
    case MRL_I16: lo = -32768.f, hi = 32767.f; break;
    case MRL_U32: return f <= 0.f ? 0u : f >= 4294967296.f ? 0xffffffffu : uint32_t(f);
    default: return f <= -2147483648.f ? 0x80000000u : f >= 2147483648.f ? 0x7fffffffu : uint32_t(int32_t(f));
  }
  f = fminf(fmaxf(f, lo), hi);
  return uint32_t(int32_t(f));
}

__device__ inline uint16_t f32_to_bf16_bits(float f) {
  uint32_t bits = __float_as_uint(f);
  if ((bits & 0x7fffffffu) > 0x7f800000u) return uint16_t((bits >> 16) | 0x40u);
  bits += 0x7fffu + ((bits >> 16) & 1u);  // round to nearest even
  return uint16_t(bits >> 16);
}

// An element's bits, zero-extended, by element size alone (no dtype switch around the load).
template <int SIZE>
__device__ inline uint32_t load_sized(const void *p, int64_t off) {
  if constexpr (SIZE == 1) return static_cast<const uint8_t *>(p)[off];
  else if constexpr (SIZE == 2) return static_cast<const uint16_t *>(p)[off];
  else return static_cast<const uint32_t *>(p)[off];
}
template <int SIZE>
__device__ inline void store_sized(void *p, int64_t off, uint32_t v) {
  if constexpr (SIZE == 1) static_cast<uint8_t *>(p)[off] = uint8_t(v);
  else if constexpr (SIZE == 2) static_cast<uint16_t *>(p)[off] = uint16_t(v);
  else static_cast<uint32_t *>(p)[off] = v;
}

// The same conversions on an element already in a register (`raw`: its bits, zero-extended).
__device__ inline float raw_to_f32(uint32_t raw, int dtype) {
  switch (dtype) {
    case MRL_U8: return float(raw & 0xffu);
    case MRL_I8: return float(int8_t(uint8_t(raw)));
    case MRL_U16: return float(raw & 0xffffu);
    case MRL_I16: return float(int16_t(uint16_t(raw)));
    case MRL_U32: return float(raw);
    case MRL_I32: return float(int32_t(raw));
    case MRL_F32: return __uint_as_float(raw);
    default: return bf16_bits_to_f32(uint16_t(raw));
  }
}
__device__ inline uint32_t convert_raw(uint32_t raw, int sdt, int ddt) {
  if (sdt == ddt) return raw;
  const bool src_float = sdt == MRL_F32 || sdt == MRL_BF16;
  if (ddt == MRL_F32) return __float_as_uint(raw_to_f32(raw, sdt));
  if (ddt == MRL_BF16) return f32_to_bf16_bits(raw_to_f32(raw, sdt));
  if (src_float) return float_to_int(raw_to_f32(raw, sdt), ddt);
  return narrow_int(sdt, raw);  // int -> int: extend by the source's sign, the store truncates
}

// Calls f(source dtype, destination dtype) with the two as compile-time constants
// (std::integral_constant), chosen once by a switch over the dtypes of SE and of DE bytes: inside
// f a conversion is the few instructions it needs, where a switch around every element costs more
// than the conversion (u8 -> bf16 over 64 Mi elements: 60 us that way, 30 this way).
template <int SE, int DE, class F>
__device__ inline void with_dtypes(int sdt, int ddt, F &&f) {
  // (u, i) of one and four bytes, (u, i, bf16) of two
  constexpr int S0 = SE == 1 ? MRL_U8 : SE == 2 ? MRL_U16 : MRL_U32, S1 = S0 + 1, S2 = SE == 2 ? MRL_BF16 : MRL_F32;
  constexpr int D0 = DE == 1 ? MRL_U8 : DE == 2 ? MRL_U16 : MRL_U32, D1 = D0 + 1, D2 = DE == 2 ? MRL_BF16 : MRL_F32;
  const int si = sdt == S0 ? 0 : sdt == S1 ? 1 : 2, di = ddt == D0 ? 0 : ddt == D1 ? 1 : 2;
#define MRL_CASE(A, B)                                                                   \
  case A * 3 + B:                                                                        \
    f(std::integral_constant<int, (A == 0 ? S0 : A == 1 ? S1 : S2)>{},                  \
      std::integral_constant<int, (B == 0 ? D0 : B == 1 ? D1 : D2)>{});                 \
    break;
  switch (si * 3 + di) {
    MRL_CASE(0, 0) MRL_CASE(0, 1) MRL_CASE(0, 2) MRL_CASE(1, 0) MRL_CASE(1, 1) MRL_CASE(1, 2)
    MRL_CASE(2, 0) MRL_CASE(2, 1) MRL_CASE(2, 2)
  }
#undef MRL_CASE
}

typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u_t __attribute__((ext_vector_type(4)));

__device__ inline uint32_t div_small(uint32_t n, uint32_t d, uint32_t inv) {
  return d == 1 ? n : __umulhi(n, inv);
}

// Coordinates of this workgroup's tile: the offsets of its origin on the two sides, and how much of
// each digit is left from there on.
// DIAGONAL: the tiles are numbered along the third digit before the second, each row of them one further on.
template <bool DIAGONAL = false>
__device__ inline void tile_origin(const MoveTile &p, int64_t &base_s, int64_t &base_d, uint32_t (&room)[MOVE_MAX_RANK]) {
  uint32_t blk = blockIdx.x;
  base_s = base_d = 0;
#pragma unroll
  for (uint32_t o = 0; o < MOVE_MAX_RANK; o++) {
    const uint32_t d = DIAGONAL && (o == 1 || o == 2) ? 3 - o : o;
    const uint32_t rest = p.by_chunks[d].div(blk);
    uint32_t at = blk - rest * p.chunks[d];
    if (DIAGONAL && d == 2) {   // (the second digit's place is the next remainder)
      at += rest - p.by_chunks[1].div(rest) * p.chunks[1];
      at -= p.by_chunks[2].div(at) * p.chunks[2];
    }
    const uint32_t origin = at * p.ext[d];
    blk = rest;
    room[d] = p.shape[d] - origin;
    base_s += int64_t(origin) * p.ss[d], base_d += int64_t(origin) * p.ds[d];
  }
}

// V elements of `size` bytes as zero-extended values <-> memory, one access of V * size bytes.
// (32 bytes, eight 32-bit values: two accesses)
template <int SIZE, int V>
__device__ inline void load_run(const void *p, int64_t off, uint32_t (&raw)[V]) {
  constexpr int BYTES = SIZE * V;
  if constexpr (V == 1 || BYTES < 4) {
#pragma unroll
    for (int e = 0; e < V; e++) raw[e] = load_sized<SIZE>(p, off + e);
  } else if constexpr (BYTES == 32) {   // two of 16, at their alignment
    const v4u_t *at = reinterpret_cast<const v4u_t *>(static_cast<const uint8_t *>(p) + off * SIZE);
    const v4u_t lo = at[0], hi = at[1];
#pragma unroll
    for (int e = 0; e < V; e++) raw[e] = e < 4 ? lo[e] : hi[e - 4];
  } else {
    typedef uint32_t W __attribute__((ext_vector_type(BYTES / 4 == 1 ? 2 : BYTES / 4)));
    const uint8_t *at = static_cast<const uint8_t *>(p) + off * SIZE;
    uint32_t w[BYTES / 4];
    if constexpr (BYTES == 4) w[0] = *reinterpret_cast<const uint32_t *>(at);
    else {
      const W v = *reinterpret_cast<const W *>(at);
#pragma unroll
      for (int i = 0; i < BYTES / 4; i++) w[i] = v[i];
    }
#pragma unroll
    for (int e = 0; e < V; e++)
      raw[e] = SIZE == 4 ? w[e] : (w[e * SIZE / 4] >> (8 * (e * SIZE % 4))) & (SIZE == 1 ? 0xffu : 0xffffu);
  }
}
template <int SIZE, int V>
__device__ inline void store_run(void *p, int64_t off, const uint32_t (&v)[V]) {
  constexpr int BYTES = SIZE * V;
  if constexpr (V == 1 || BYTES < 4) {
#pragma unroll
    for (int e = 0; e < V; e++) store_sized<SIZE>(p, off + e, v[e]);
  } else {
    uint32_t w[BYTES / 4];
#pragma unroll
    for (int i = 0; i < BYTES / 4; i++) w[i] = 0;
#pragma unroll
    for (int e = 0; e < V; e++) {
      if constexpr (SIZE == 4) w[e] = v[e];
      else w[e * SIZE / 4] |= (v[e] & (SIZE == 1 ? 0xffu : 0xffffu)) << (8 * (e * SIZE % 4));
    }
    uint8_t *at = static_cast<uint8_t *>(p) + off * SIZE;
    if constexpr (BYTES == 4) MRL_STORE_ONCE(w[0], reinterpret_cast<uint32_t *>(at));
    else if constexpr (BYTES == 8) MRL_STORE_ONCE((v2u{w[0], w[1]}), reinterpret_cast<v2u *>(at));
    else MRL_STORE_ONCE((v4u_t{w[0], w[1], w[2], w[3]}), reinterpret_cast<v4u_t *>(at));
  }
}

}  // namespace
}  // namespace mrl
