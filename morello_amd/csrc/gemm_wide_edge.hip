// The four-wave 256 x 256 tile (gemm_wide_kernel.h) on any M and N and against a k-fastest B, in a translation unit
// of its own: each of its instantiations is four bodies of assembly.
#include "gemm_wide_kernel.h"

namespace mrl {
using namespace gemm;

hipError_t launch_gemm_wide_edge(const GemmArgs &g, int kind, hipStream_t stream) {
  switch (kind) {
    case 0: return g.b_kmajor ? launch_wide<I8, false, true, true>(g, stream) : launch_wide<I8, false, false, true>(g, stream);
    case 1: return g.b_kmajor ? launch_wide<I8, true, true, true>(g, stream) : launch_wide<I8, true, false, true>(g, stream);
    case 2: return g.b_kmajor ? launch_wide<BF16, false, true, true>(g, stream) : launch_wide<BF16, false, false, true>(g, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mrl
