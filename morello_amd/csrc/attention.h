// What the two forms of the fused Matmul -> Softmax -> Matmul share (attention.hip, attention_keys.hip).
#pragma once
#include "kernels.h"

namespace mrl {
namespace attn {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4s lds_v4s;
typedef __attribute__((address_space(3))) void lds_void;

constexpr float LOG2E = 1.44269504088896340736f;
constexpr float STALE_REFERENCE = 1.0e12f;  // ~2^40: an exponential beyond it moves the reference
// The reference before the first block: below any score, and its multiple by log2 e is still finite (a block of keys
// that all score -inf has exponentials of 0, not of inf - inf).
constexpr float NO_REFERENCE = -2.0e38f;
constexpr uint32_t OUTSIDE = 0x80000000u;   // an offset no resource here holds, whatever block's is added

// One direct-to-LDS load: 64 lanes x 16 bytes from `base + voff` (voff per lane) to the 1 KiB at
// LDS address `lds_addr` (wave-uniform), lane l to slot l.  Written as assembly so that the
// compiler does not know of it: it would otherwise make every later LDS read wait for all such
// loads in flight (it cannot tell the stages apart), which serialises a block's softmax behind
// the next block's fetch.  The waits that matter are the explicit ones before the barriers.
__device__ inline void dma16(const uint8_t *base, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(voff), "s"(base));
}
// The same through a buffer resource: an offset past its end brings zeros.
__device__ inline void dma16(__amdgpu_buffer_rsrc_t from, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" : : "s"(lds_addr), "v"(voff), "s"(from));
}
// The same where no barrier stands between the reads of what was in LDS and the load that replaces it: no read is
// moved past it by the compiler.
__device__ inline void dma16_ordered(__amdgpu_buffer_rsrc_t from, uint32_t voff, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" : : "s"(lds_addr), "v"(voff), "s"(from) : "memory");
}
__device__ inline uint32_t lds_address(const void *p) {
  return uint32_t(reinterpret_cast<uintptr_t>((lds_void *)p));
}

__device__ inline v2i read_tr16(const uint8_t *p) {
  const v4s r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)p);
  return __builtin_bit_cast(v2i, r);
}

}  // namespace attn
}  // namespace mrl
