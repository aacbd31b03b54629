// Host check of how f32 Matmuls share K out (morello_amd/csrc/gemm_f32.hip): the kernels' first step loads 32 of K whatever is left of it, so
// that no slice may be shorter, for any K and number of slices and for those that the rule picks.  Nothing is launched.
#include <cstdio>

#include "../morello_amd/csrc/kernels.h"

int main() {
  int bad = 0, sliced = 0;
  auto check = [&](uint32_t k, uint32_t slice_k, uint32_t m, uint32_t n) {
    const uint32_t last = k % slice_k == 0 ? slice_k : k % slice_k;
    if (slice_k % 32 != 0 || slice_k < 128 || last < 32) bad++, std::printf("%u x %u x %u in slices of %u, the last of %u\n", m, k, n, slice_k, last);
  };
  for (uint32_t k = 16; k <= 40000; k++)
    for (uint32_t want = 2; want <= 16; want++)
      if (const uint32_t slice_k = mrl::gemm_f32_slice_k(k, want); slice_k != 0 && slice_k < k) check(k, slice_k, 0, 0);
  const uint32_t sides[][2] = {{48, 1040}, {272, 304}, {400, 272}, {112, 464}, {144, 304}, {112, 144}, {720, 16}, {64, 1056}, {128, 544}, {128, 1088}, {33, 97}, {537, 569}, {256, 256}, {640, 640}};
  for (uint32_t k = 16; k <= 12000; k++)
    for (const auto &side : sides)
      for (bool b_kmajor : {false, true}) {
        mrl::GemmArgs g;
        g.a = reinterpret_cast<const void *>(uintptr_t(1) << 20), g.b = reinterpret_cast<const void *>(uintptr_t(2) << 20), g.c = reinterpret_cast<void *>(uintptr_t(3) << 20);
        g.batch = 1, g.m = side[0], g.n = side[1], g.k = k, g.b_kmajor = b_kmajor;
        g.lda = k, g.ldb = b_kmajor ? k : g.n, g.ldc = g.n, g.sa = g.sb = g.sc = 0, g.accum = 0;
        uint32_t slice_k = 0;
        const uint32_t count = mrl::gemm_f32_slices(g, &slice_k);
        if (count == 1) continue;
        sliced++;
        if (count != (k + slice_k - 1) / slice_k) bad++, std::printf("%u x %u x %u: %u slices of %u\n", g.m, k, g.n, count, slice_k);
        check(k, slice_k, g.m, g.n);
      }
  if (sliced < 100000) bad++, std::printf("only %d problems in slices\n", sliced);
  if (bad == 0) std::printf("f32 slices ok\n");
  return bad != 0;
}
