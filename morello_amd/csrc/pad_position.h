// Which bytes of a source row a 16-byte chunk of its padded copy holds.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define MRL_PAD_HD __host__ __device__
#else
#define MRL_PAD_HD
#endif

namespace mrl {

struct PadChunk {
  int64_t at;   // the first of them, in bytes from the row's start; 0 where there are none
  int left;     // how many: 0 .. 16
};
// The `chunk`-th chunk of a row of `row_bytes`.  64 bits throughout: a row of 2^31 - 1 elements is up to 8 GiB
// long.
MRL_PAD_HD inline PadChunk pad_chunk(uint32_t chunk, uint64_t row_bytes) {
  const uint64_t at = uint64_t(chunk) * 16;
  if (at >= row_bytes) return {0, 0};
  return {int64_t(at), row_bytes - at < 16 ? int(row_bytes - at) : 16};
}

}  // namespace mrl
