// Host check of the Matmul dispatch (morello_amd/csrc/gemm_mfma.hip) on addresses: which outputs the matrix-core kernels
// take.  Nothing is launched; the addresses are made up.
#include <cstdio>
#include <initializer_list>

#include "../morello_amd/csrc/kernels.h"

static mrl::GemmArgs args(uintptr_t c, bool c_bf16) {
  mrl::GemmArgs g;
  g.a = reinterpret_cast<const void *>(uintptr_t(1) << 20), g.b = reinterpret_cast<const void *>(uintptr_t(2) << 20);
  g.c = reinterpret_cast<void *>((uintptr_t(3) << 20) + c);
  g.batch = 1, g.m = 1000, g.n = 1024, g.k = 2048;
  g.lda = 2048, g.ldb = 1024, g.ldc = 1024;
  g.sa = g.sb = g.sc = 0, g.accum = 0, g.c_bf16 = c_bf16;
  return g;
}

int main() {
  int bad = 0;
  for (uintptr_t at = 0; at < 8; at++) {
    if (mrl::gemm_possible(args(at, true), 2) != (at % 2 == 0)) bad++, std::printf("bf16 C at %d\n", int(at));
    if (mrl::gemm_possible(args(at, false), 2) != (at % 4 == 0)) bad++, std::printf("f32 C at %d\n", int(at));
    // one row against a large k-fastest B: the dot products
    for (bool c_bf16 : {true, false}) {
      mrl::GemmArgs row = args(at, c_bf16);
      row.m = 1, row.n = 12000, row.ldb = 2048, row.ldc = 12000, row.b_kmajor = true;
      if (mrl::gemv_applicable(row, 2) != (at % (c_bf16 ? 2 : 4) == 0)) bad++, std::printf("dot products, C at %d\n", int(at));
    }
  }
  if (bad == 0) std::printf("dispatch ok\n");
  return bad != 0;
}
