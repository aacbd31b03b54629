// Sixteen bytes at any address out of aligned loads.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mrl {

typedef int chunk_t __attribute__((ext_vector_type(4)));

// The sixteen bytes from byte `shift` (0 .. 15) of two chunks on.
__device__ inline chunk_t cut_chunk(chunk_t lo, chunk_t hi, uint32_t shift) {
  // by one and by two words as bit selects (as conditional copies the compiler moves the words
  // through LDS), then by bytes
  const uint32_t by1 = 0u - (shift >> 2 & 1), by2 = 0u - (shift >> 3 & 1);
  uint32_t t[8] = {uint32_t(lo[0]), uint32_t(lo[1]), uint32_t(lo[2]), uint32_t(lo[3]),
                   uint32_t(hi[0]), uint32_t(hi[1]), uint32_t(hi[2]), uint32_t(hi[3])};
#pragma unroll
  for (int i = 0; i < 7; i++) t[i] = (t[i + 1] & by1) | (t[i] & ~by1);
#pragma unroll
  for (int i = 0; i < 5; i++) t[i] = (t[i + 2] & by2) | (t[i] & ~by2);
  chunk_t v;
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = int(__builtin_amdgcn_alignbyte(t[i + 1], t[i], shift & 3));
  return v;
}

// The first `left` bytes of v, zeros behind them.
__device__ inline chunk_t keep_bytes(chunk_t v, int left) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int n = left - 4 * i;
    v[i] &= n >= 4 ? -1 : n <= 0 ? 0 : int((1u << (8 * n)) - 1);
  }
  return v;
}

}  // namespace mrl
