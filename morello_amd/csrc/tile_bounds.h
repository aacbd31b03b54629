// How much of a row-major right operand a tile's loads may touch.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define MRL_BOUNDS_HD __host__ __device__
#else
#define MRL_BOUNDS_HD
#endif

namespace mrl {

// Bytes from a tile's first column on, of `rows` rows `ld_bytes` apart: up to the end of the 16-byte chunk that holds the last
// row's last column of the tile, `column_bytes` from the first.  (Not up to that row's end: where the rows of several batch entries lie between
// each other, [k][batch][n] in memory, what follows the last entry's last row up to its leading dimension is nobody's.)
MRL_BOUNDS_HD inline int64_t tile_bytes(int64_t rows, int64_t ld_bytes, int64_t column_bytes) {
  return (rows - 1) * ld_bytes + (column_bytes + 15) / 16 * 16;
}

}  // namespace mrl
