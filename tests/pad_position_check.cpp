// Host check of morello_amd/csrc/pad_position.h: the chunks of a row take its bytes one after the other, each
// byte once and none outside, for rows on either side of 2^31 and 2^32 bytes.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "../morello_amd/csrc/pad_position.h"

static void check(uint64_t row_bytes, uint64_t chunk) {
  const mrl::PadChunk c = mrl::pad_chunk(uint32_t(chunk), row_bytes);
  const uint64_t at = chunk * 16, want = at >= row_bytes ? 0 : row_bytes - at < 16 ? row_bytes - at : 16;
  const bool ok = uint64_t(c.left) == want && c.at == int64_t(want ? at : 0) && c.at >= 0 && uint64_t(c.at) + uint64_t(c.left) <= row_bytes;
  if (ok) return;
  std::printf("row of %llu bytes, chunk %llu: %d bytes at %lld\n", (unsigned long long)row_bytes, (unsigned long long)chunk, c.left, (long long)c.at);
  std::exit(1);
}

int main() {
  const uint64_t around[] = {16, 1024, 1ull << 31, 2400000004ull, 1ull << 32, (1ull << 33) - 64};
  for (uint64_t middle : around)
    for (int64_t d = -17; d <= 17; d++) {
      const uint64_t row_bytes = middle + uint64_t(d);
      if (int64_t(row_bytes) <= 0) continue;
      const uint64_t chunks = (row_bytes + 15) / 16;
      for (uint64_t c : {uint64_t(0), uint64_t(1), chunks / 2, (uint64_t(1) << 27) - 1, uint64_t(1) << 27, chunks - 1, chunks, chunks + 7})
        if (c < (uint64_t(1) << 32)) check(row_bytes, c);
    }
  std::printf("pad positions ok\n");
}
