// Host check of morello_amd/csrc/tile_bounds.h: what the tiles' loads of a row-major right operand reach when rows
// of several batch entries lie between each other ([k][batch][n] in memory), and of rows one after the other.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "../morello_amd/csrc/tile_bounds.h"

// Tiles of `bn` columns in steps of 128 bytes of K over the last batch entry of [k][batch][n] elements of `es` bytes.
static void check(int64_t es, int64_t bn, int64_t k, int64_t batch, int64_t n) {
  const int64_t bk = 128 / es, ld_bytes = batch * n * es, entry = (batch - 1) * n * es, operand = k * ld_bytes;
  for (int64_t n0 = 0; n0 < n; n0 += bn)
    for (int64_t k0 = 0; k0 < k; k0 += bk) {
      const int64_t rows = k - k0 < bk ? k - k0 : bk, columns = n - n0 < bn ? n - n0 : bn;
      const int64_t from = entry + k0 * ld_bytes + n0 * es, bytes = mrl::tile_bytes(rows, ld_bytes, columns * es);
      for (int64_t r = 0; r < bk; r++)
        for (int64_t c = 0; c < bn * es; c += 16) {   // a load: 16 bytes, all of them inside the resource or zeros
          const int64_t at = r * ld_bytes + c;
          const bool loaded = at + 16 <= bytes, wanted = r < rows && c < columns * es;
          // past K or the operand's end nothing may be touched; what is multiplied has to be there
          if ((!loaded || (r < rows && from + at + 16 <= operand)) && (loaded || !wanted)) continue;
          std::printf("es %lld, tiles of %lld, %lld x %lld x %lld: row %lld of %lld, byte %lld: %lld past the operand\n", (long long)es,
                      (long long)bn, (long long)batch, (long long)k, (long long)n, (long long)r, (long long)rows, (long long)c,
                      (long long)(from + at + 16 - operand));
          std::exit(1);
        }
    }
}

int main() {
  for (int64_t es : {1, 2, 4})
    for (int64_t bn : {64, 128, 160, 192, 256})
      for (int64_t batch : {1, 2, 3})
        for (int64_t chunks : {1, 3, 5, 9, 13, 17, 24})   // of 16 bytes: N on both sides of whole tiles
          for (int64_t k : {1, 15, 32, 70, 128, 131}) check(es, bn, k, batch, chunks * 16 / es);
  std::printf("tile bounds ok\n");
}
