// Conv NHWC u8|i8 x KRSC i8 -> i32 and bf16 x bf16 -> f32 for pixels of three or four channels (a first
// layer), channels-last (morello/src/spec.rs:486-494: no stride, no padding): the form of
// conv_windows.hip's kernel that needs no windows in LDS.
//
// What bounds such a layer is its output (16 x 109 x 109 x 64 floats: 49 MB against 1 MB of image) as long as
// nothing else takes time; the other form's chain of patch, barrier, copied windows, barrier, MFMAs per
// 128 pixels did (that layer in bf16, 7 x 7: 27.5 us).  Here a pixel takes four elements in LDS,
// the fourth zero if there are three, so a window's row is a run of whole pixels at an address a
// multiple of the pixel apart and MFMA operands are read where they lie:
//   - a row of a window is 1, 2 or 4 chunks of 16 bytes (cpr; three are taken as four), a k step of 64
//     bytes is 4 / cpr rows, and what a lane reads for step s lies s * 4 / cpr patch rows below what it
//     reads for step 0: one address per lane, whatever the filter's size;
//   - a wave works alone on 16 x 2 output pixels, its patch in LDS of its own: no barrier after the
//     filters are staged.  The next item's pixels are fetched while this one is multiplied;
//   - filters lie in the same order, zeros wherever no pixel is.  Floats: window positions
//     past the filter's width or height are zeroed as well (a NaN there times zero is not zero).
// A lane holds four consecutive filters of a pixel: 16 bytes, four lanes 64 contiguous ones, and two
// such stores fill a cache line: they go through the L2 (past it, 32 x 3 -> 96 x 224 x 224 took 209 us).
// Measured, the other form / this (us, TB/s of image, filters and output): bf16 7 x 7 16 x 3 -> 64 x 109^2 28.1 / 17.0,
// 2.9; 32 x 3 -> 96 x 224^2 298 / 146, 4.3; 1 x 3 -> 64 x 109^2 10.4 / 5.4; 3 x 3 32 x 4 -> 16 x 224^2 80 / 23, 5.0; u8 7 x 7
// 16 x 3 -> 64 x 109^2 23.0 / 15.1.  Items of four rows: 1 x 3 -> 64 x 109^2 6.9, 3 x 3 22.1, the others within 3 %.
#include <algorithm>

#include "kernels.h"
#include "plan.h"

namespace mrl {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
enum { IMG_I8 = 0, IMG_U8 = 1, IMG_BF16 = 2 };

constexpr int WAVES = 8, ITEM_W = 16, ITEM_H = 2;
constexpr int HELD = 4;   // patch pixels a lane holds in flight
constexpr int STRIP_CHUNKS = 6;   // of 64 pixels that a strip's patch may be
constexpr int FB = 2;     // blocks of 16 filters multiplied at a time

struct PixelsArgs {
  const uint8_t *image, *filters;
  int32_t *out;
  uint32_t f, oh, ow, h, w, fh, fw;
  uint32_t group;               // filters a workgroup takes, a multiple of 32
  uint32_t pixel_bytes;         // of a pixel in memory: 3 or 4 elements
  int accum;
  uint32_t items, steps;        // 16 x 2 pieces of the output; k steps (KS whole ones and perhaps a tail)
  uint32_t chunks_log2;         // log2 of cpr
  uint32_t slots;               // pixels of a filter's row in LDS: steps * 64 / PB
  uint32_t patch_w, patch_h;    // pixels
  int whole_lines;              // 32 filters of a pixel are a cache line of the output
  uint32_t patch_bytes;         // of LDS, rows that only a tail step's masked lanes read included
  FastDiv by_image, by_row, by_slots, by_patch_w;   // items of an image, of an image's row of them
  uint32_t strip, per_image, image_bytes;           // strips: output rows of one, strips and bytes of an image
};

// Pixels of four elements in LDS out of pixels of three or four in memory.
template <int KIND>
struct Pixels {
  static constexpr bool HALVES = KIND == IMG_BF16;
  static constexpr int ES = HALVES ? 2 : 1, PB = 4 * ES, PER_CHUNK = 16 / PB;   // bytes of a pixel in LDS, pixels of a chunk
  typedef typename std::conditional<HALVES, float, int>::type Element;
  typedef Element Acc __attribute__((ext_vector_type(4)));
  struct Pixel { uint32_t v[ES]; };
  struct Raw { uint32_t v[ES + 1]; uint32_t shift; };
  __device__ static Acc mfma(v4i a, v4i b, Acc c) {
    if constexpr (HALVES) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
  // A pixel out of the aligned dwords it lies in (a dword without a byte of it is not read).
  __device__ static Raw fetch(const uint8_t *at, uint32_t pixel_bytes) {
    Raw r;
    r.shift = uint32_t(reinterpret_cast<uintptr_t>(at)) & 3;
    const uint32_t *from = reinterpret_cast<const uint32_t *>(at - r.shift);
#pragma unroll
    for (int i = 0; i < ES; i++) r.v[i] = from[i];
    r.v[ES] = from[r.shift + pixel_bytes > 4 * ES ? ES : ES - 1];
    return r;
  }
  __device__ static Pixel pixel(const Raw &r, uint32_t pixel_bytes) {
    const uint32_t last_mask = pixel_bytes == PB ? 0xffffffffu : HALVES ? 0xffffu : 0xffffffu;
    Pixel x;
#pragma unroll
    for (int i = 0; i < ES; i++) x.v[i] = __builtin_amdgcn_alignbyte(r.v[i + 1], r.v[i], r.shift);
    x.v[ES - 1] &= last_mask;
    return x;
  }
  __device__ static void put(uint8_t *to, const Pixel &x) {
    if constexpr (HALVES) *(v2u *)to = v2u{x.v[0], x.v[ES - 1]};
    else *(uint32_t *)to = x.v[0];
  }
  // The image's pixels as they are multiplied: u8 as a - 128.
  __device__ static void put_image(uint8_t *to, const Raw &r, uint32_t pixel_bytes) {
    Pixel x = pixel(r, pixel_bytes);
    if (KIND == IMG_U8) x.v[0] ^= 0x80808080u;
    put(to, x);
  }
  // This workgroup's filters, `nf` from f0 on, into rows of `filter_row` bytes at `filt` (`group` of them, zeros where no pixel
  // is): their bytes are one contiguous piece of memory, fetched in whole chunks with the loads in flight together into
  // the LDS behind, then spread out pixel by pixel.  ONE_BATCH: no more than the loop's first round
  // (32 filters are 12 KiB), whose loads are otherwise made to wait for a patch in flight.
  template <bool ONE_BATCH = false>
  __device__ static void stage_filters(const PixelsArgs &p, uint32_t group, uint32_t f0, uint32_t nf, uint32_t filter_row, uint8_t *filt) {
    const int tid = threadIdx.x;
    const uint32_t filter_bytes = p.fh * p.fw * p.pixel_bytes;
    const uint8_t *from = p.filters + uint64_t(f0) * filter_bytes;
    const uint32_t head = uint32_t(reinterpret_cast<uintptr_t>(from)) & 15, chunks = (head + nf * filter_bytes + 15) / 16;
    const v4i *first = reinterpret_cast<const v4i *>(from - head);
    v4i *raw = reinterpret_cast<v4i *>(filt + group * filter_row);
    constexpr uint32_t BATCH = 3;
    for (uint32_t c0 = 0; c0 < chunks; c0 += BATCH * 64 * WAVES) {
      v4i got[BATCH];
#pragma unroll
      for (uint32_t j = 0; j < BATCH; j++) got[j] = first[min(c0 + j * 64 * WAVES + tid, chunks - 1)];
#pragma unroll
      for (uint32_t j = 0; j < BATCH; j++)
        if (c0 + j * 64 * WAVES + tid < chunks) raw[c0 + j * 64 * WAVES + tid] = got[j];
      if (ONE_BATCH) break;
    }
    __syncthreads();
    const uint32_t *words = reinterpret_cast<const uint32_t *>(raw);
    const uint32_t per_row = uint32_t(PER_CHUNK) << p.chunks_log2;   // pixels a window's row takes
#pragma unroll 2
    for (uint32_t i = tid; i < group * p.slots; i += 64 * WAVES) {
      const uint32_t fi = p.by_slots.div(i), s = i - fi * p.slots;
      const uint32_t r = s / PER_CHUNK >> p.chunks_log2, x = s & (per_row - 1);
      const bool real = fi < nf && r < p.fh && x < p.fw;
      const uint32_t at = real ? head + ((fi * p.fh + r) * p.fw + x) * p.pixel_bytes : head;
      Raw px;
#pragma unroll
      for (int w = 0; w <= ES; w++) px.v[w] = words[at / 4 + w];
      px.shift = at & 3;
      put(filt + fi * filter_row + s * PB, real ? pixel(px, p.pixel_bytes) : Pixel{});
    }
    __syncthreads();   // the raw bytes are no longer needed
  }
};

// KS: whole k steps of 64 bytes (a window's chunks / 4); the rest is a tail whose lanes past the
// filter's last row count for nothing.  PIXELS: always true; tells this form from the other one in plans and profiles.
template <int KS, int KIND, bool PIXELS>
__global__ __launch_bounds__(64 * WAVES, 4) void k_conv_windows(PixelsArgs p) {
  typedef Pixels<KIND> P;
  typedef typename P::Acc Acc;
  typedef typename P::Raw Raw;
  constexpr bool HALVES = P::HALVES;
  constexpr int PB = P::PB, PER_CHUNK = P::PER_CHUNK;
  extern __shared__ __attribute__((aligned(16))) uint8_t pix_lds[];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t filter_row = p.steps * 64 + 16;   // 16 bytes more than the length: spreads an operand read over the banks
  uint8_t *filt = pix_lds;
  uint8_t *patch = pix_lds + p.group * filter_row + wave * p.patch_bytes;
  const uint32_t f0 = blockIdx.y * p.group, nf = min(p.group, p.f - f0);   // this workgroup's filters (a multiple of 16)

  // Where in a patch a lane's held pixels are does not depend on the item.
  uint32_t held_y[HELD], held_x[HELD];
  const uint32_t patch_pixels = p.patch_w * p.patch_h;
#pragma unroll
  for (int j = 0; j < HELD; j++) {
    const uint32_t i = lane + j * 64;
    held_y[j] = p.by_patch_w.div(i), held_x[j] = i - held_y[j] * p.patch_w;
  }
  struct Corner { uint32_t img, y0, x0; };
  const uint32_t tiles_x = (p.ow + ITEM_W - 1) / ITEM_W, per_image = tiles_x * ((p.oh + ITEM_H - 1) / ITEM_H);
  auto corner_of = [&](uint32_t item) {
    const uint32_t img = p.by_image.div(item), in_img = item - img * per_image, ty = p.by_row.div(in_img);
    return Corner{img, ty * ITEM_H, (in_img - ty * tiles_x) * ITEM_W};
  };
  // (past the image's edge, its last row or pixel again: those reach only results that are not
  // stored, or positions past the filter's width)
  auto source = [&](const Corner &at, uint32_t r, uint32_t x) {
    return p.image + ((uint64_t(at.img) * p.h + min(at.y0 + r, p.h - 1)) * p.w + min(at.x0 + x, p.w - 1)) * p.pixel_bytes;
  };
  Raw held[HELD];
  auto fetch_patch = [&](const Corner &at) {
#pragma unroll
    for (int j = 0; j < HELD; j++)
      if (lane + j * 64 < int(patch_pixels)) held[j] = P::fetch(source(at, held_y[j], held_x[j]), p.pixel_bytes);
  };
  const uint32_t stride = gridDim.x * WAVES;
  uint32_t item = blockIdx.x * WAVES + wave;
  if (item < p.items) fetch_patch(corner_of(item));   // in flight while the filters are staged
  P::stage_filters(p, p.group, f0, nf, filter_row, filt);   // (the bytes as they lie in memory into what will be the patches)
  const uint8_t *my_filt = filt + li * filter_row + lg * 16;
  // u8 pixels are multiplied as a - 128: 128 times a filter's sum comes on top (kept in LDS, in the
  // 16 bytes between the filters' rows).
  if constexpr (KIND == IMG_U8) {
    const v4i ones = v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101};
    for (uint32_t fb = wave; fb < p.group / 16; fb += WAVES) {
      Acc sum = {};
      for (uint32_t ks = 0; ks < p.steps; ks++) sum = P::mfma(*(const v4i *)(my_filt + fb * 16 * filter_row + ks * 64), ones, sum);
      if (li == 0) *(v4i *)(filt + (fb * 16 + lg) * filter_row + p.steps * 64) = sum * 128;
    }
    __syncthreads();
  }
  // This lane's chunk of a step: row lg / cpr of the step's, chunk lg % cpr of the row.
  const uint32_t row_bytes = p.patch_w * PB, chunk = lg & ((1u << p.chunks_log2) - 1), row_of = uint32_t(lg) >> p.chunks_log2;
  const uint32_t step_bytes = (4u >> p.chunks_log2) * row_bytes;
  const uint8_t *my_patch = patch + row_of * row_bytes + li * PB + chunk * 16;
  const uint32_t keep_lo = chunk * PER_CHUNK < p.fw ? 0xffffffffu : 0u, keep_hi = chunk * PER_CHUNK + 1 < p.fw ? 0xffffffffu : 0u;
  auto window = [&](uint32_t ks, int pb) {
    const uint8_t *at = my_patch + ks * step_bytes + pb * row_bytes;
    if constexpr (HALVES) {
      const v2u lo = *(const v2u *)at & keep_lo, hi = *(const v2u *)(at + 8) & keep_hi;
      return v4i{int(lo[0]), int(lo[1]), int(hi[0]), int(hi[1])};
    } else {
      const uint32_t *w = (const uint32_t *)at;
      return v4i{int(w[0]), int(w[1]), int(w[2]), int(w[3])};
    }
  };
  for (; item < p.items; item += stride) {
    const Corner at = corner_of(item);
#pragma unroll
    for (int j = 0; j < HELD; j++)
      if (lane + j * 64 < int(patch_pixels)) P::put_image(patch + (lane + j * 64) * PB, held[j], p.pixel_bytes);
    for (uint32_t i = lane + HELD * 64; i < patch_pixels; i += 64) {
      const uint32_t r = p.by_patch_w.div(i);
      P::put_image(patch + i * PB, P::fetch(source(at, r, i - r * p.patch_w), p.pixel_bytes), p.pixel_bytes);
    }
    // The wave's LDS accesses complete in order: what is left is that the compiler keeps them so.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (item + stride < p.items) fetch_patch(corner_of(item + stride));
    // Two blocks of filters at a time: with four at once the registers of half as many waves.
#pragma unroll 1
    for (uint32_t fb0 = 0; fb0 < nf; fb0 += 16 * FB) {
      asm volatile("" : : : "memory");   // (else the window operands of all steps are kept from pass to pass, and spill)
      Acc acc[ITEM_H][FB];
#pragma unroll
      for (int fb = 0; fb < FB; fb++) {
        Acc from = {};
        if constexpr (KIND == IMG_U8) from = *(const v4i *)(filt + (fb0 + fb * 16 + lg) * filter_row + p.steps * 64);
#pragma unroll
        for (int pb = 0; pb < ITEM_H; pb++) acc[pb][fb] = from;
      }
      const uint8_t *block = my_filt + fb0 * filter_row;
      auto step = [&](uint32_t ks, bool inside) {
        v4i a[FB], bop[ITEM_H];
#pragma unroll
        for (int fb = 0; fb < FB; fb++) a[fb] = *(const v4i *)(block + fb * 16 * filter_row + ks * 64);
#pragma unroll
        for (int pb = 0; pb < ITEM_H; pb++) {
          bop[pb] = window(ks, pb);
          if (HALVES && !inside) bop[pb] = v4i{0, 0, 0, 0};
        }
#pragma unroll
        for (int pb = 0; pb < ITEM_H; pb++)
#pragma unroll
          for (int fb = 0; fb < FB; fb++) acc[pb][fb] = P::mfma(a[fb], bop[pb], acc[pb][fb]);
      };
#pragma unroll 2
      for (int ks = 0; ks < KS; ks++) step(ks, true);
      if (p.steps > KS) step(KS, KS * (4u >> p.chunks_log2) + row_of < p.fh);
      const uint32_t x = at.x0 + li;
#pragma unroll
      for (int pb = 0; pb < ITEM_H; pb++) {
        const uint32_t y = at.y0 + pb;
        if (y < p.oh && x < p.ow) {
          Acc *d = (Acc *)(p.out + ((uint64_t(at.img) * p.oh + y) * p.ow + x) * p.f + f0 + fb0 + 4 * lg);
#pragma unroll
          for (int fb = 0; fb < FB; fb++)
            if (fb0 + fb * 16 < nf) {
              Acc v = acc[pb][fb];
              if (p.accum) v += d[4 * fb];
              d[4 * fb] = v;
            }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// The same with the filters' operands in registers, for filters of up to seven rows whose rows are RPS to a step (1, 2 or 4):
// a workgroup takes 32 filters, and the operand of patch row r serves every pair of a step and an output row with
// RPS * step + row = r.  What bounded the form above beside its stores was LDS, 56 KB read per 16 x 2 pixels and 64 filters of bf16
// 7 x 7; here 16 KB are.  Bound now by the stores of the output and by the start (filters staged, a first patch: 4 us). us, the
// form above / this: bf16 7 x 7 16 x 3 -> 64 x 109^2 17.2 / 15.5, 32 x 3 -> 96 x 224^2 154 / 131, u8 7 x 7 12 x 4 -> 96 x 76^2 12.5 / 8.8.
template <int KS, int RPS, bool TAIL, int KIND, bool PIXELS>
__global__ __launch_bounds__(64 * WAVES, 4) void k_conv_windows(PixelsArgs p) {
  typedef Pixels<KIND> P;
  typedef typename P::Acc Acc;
  typedef typename P::Raw Raw;
  constexpr bool HALVES = P::HALVES;
  constexpr int PB = P::PB, PER_CHUNK = P::PER_CHUNK, STEPS = KS + TAIL, CHUNKS = 4 / RPS, GROUP = 16 * FB;
  constexpr uint32_t filter_row = STEPS * 64 + 16, patch_w = ITEM_W - 1 + PER_CHUNK * CHUNKS, row_bytes = patch_w * PB;
  constexpr int ROWS = RPS * (STEPS - 1) + ITEM_H;      // patch rows that operands start in
  extern __shared__ __attribute__((aligned(16))) uint8_t pix_lds[];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint8_t *const patch = pix_lds + wave * p.patch_bytes;   // (where the filters lay while they were staged)
  const uint32_t f0 = blockIdx.y * GROUP, nf = min(uint32_t(GROUP), p.f - f0);

  const uint32_t patch_pixels = patch_w * p.patch_h;
  struct Corner { uint32_t img, y0, x0; };
  const uint32_t tiles_x = (p.ow + ITEM_W - 1) / ITEM_W, per_image = tiles_x * ((p.oh + ITEM_H - 1) / ITEM_H);
  auto corner_of = [&](uint32_t item) {
    const uint32_t img = p.by_image.div(item), in_img = item - img * per_image, ty = p.by_row.div(in_img);
    return Corner{img, ty * ITEM_H, (in_img - ty * tiles_x) * ITEM_W};
  };
  auto source = [&](const Corner &at, uint32_t r, uint32_t x) {   // (past the image's edge: as above)
    return p.image + ((uint64_t(at.img) * p.h + min(at.y0 + r, p.h - 1)) * p.w + min(at.x0 + x, p.w - 1)) * p.pixel_bytes;
  };
  Raw held[HELD];
  auto fetch_patch = [&](const Corner &at) {
#pragma unroll
    for (int j = 0; j < HELD; j++) {
      const uint32_t i = lane + j * 64, r = i / patch_w;
      if (i < patch_pixels) held[j] = P::fetch(source(at, r, i - r * patch_w), p.pixel_bytes);
    }
  };
  const uint32_t stride = gridDim.x * WAVES;
  uint32_t item = blockIdx.x * WAVES + wave;
  if (item < p.items) fetch_patch(corner_of(item));   // in flight while the filters are staged
  P::stage_filters(p, GROUP, f0, nf, filter_row, pix_lds);
  v4i a[STEPS][FB];
#pragma unroll
  for (int ks = 0; ks < STEPS; ks++)
#pragma unroll
    for (int fb = 0; fb < FB; fb++) a[ks][fb] = *(const v4i *)(pix_lds + (fb * 16 + li) * filter_row + lg * 16 + ks * 64);
  Acc start[FB];   // u8 pixels are multiplied as a - 128: 128 times a filter's sum comes on top
#pragma unroll
  for (int fb = 0; fb < FB; fb++) {
    start[fb] = Acc{};
    if constexpr (KIND == IMG_U8) {
      const v4i ones = v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
      for (int ks = 0; ks < STEPS; ks++) start[fb] = P::mfma(a[ks][fb], ones, start[fb]);
      start[fb] *= 128;
    }
  }
  __syncthreads();   // every wave holds its operands: the patches may lie there
  const uint32_t chunk = lg & (CHUNKS - 1), row_of = uint32_t(lg) / CHUNKS;
  const uint8_t *my_patch = patch + row_of * row_bytes + li * PB + chunk * 16;
  const uint32_t keep_lo = chunk * PER_CHUNK < p.fw ? 0xffffffffu : 0u, keep_hi = chunk * PER_CHUNK + 1 < p.fw ? 0xffffffffu : 0u;
  const bool inside = KS * RPS + row_of < p.fh;   // of the tail step
  for (; item < p.items; item += stride) {
    const Corner at = corner_of(item);
#pragma unroll
    for (int j = 0; j < HELD; j++)
      if (lane + j * 64 < int(patch_pixels)) P::put_image(patch + (lane + j * 64) * PB, held[j], p.pixel_bytes);
    // The wave's LDS accesses complete in order: what is left is that the compiler keeps them so.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (item + stride < p.items) fetch_patch(corner_of(item + stride));
    Acc acc[ITEM_H][FB];
#pragma unroll
    for (int pb = 0; pb < ITEM_H; pb++)
#pragma unroll
      for (int fb = 0; fb < FB; fb++) acc[pb][fb] = start[fb];
#pragma unroll
    for (int r = 0; r < ROWS; r++) {
      v4i bop;
      if constexpr (HALVES) {
        const v2u lo = *(const v2u *)(my_patch + r * row_bytes) & keep_lo, hi = *(const v2u *)(my_patch + r * row_bytes + 8) & keep_hi;
        bop = v4i{int(lo[0]), int(lo[1]), int(hi[0]), int(hi[1])};
      } else {
        const uint32_t *w = (const uint32_t *)(my_patch + r * row_bytes);
        bop = v4i{int(w[0]), int(w[1]), int(w[2]), int(w[3])};
      }
#pragma unroll
      for (int ks = 0; ks < STEPS; ks++) {
        const int pb = r - RPS * ks;
        if (pb < 0 || pb >= ITEM_H) continue;
        const v4i b = HALVES && TAIL && ks == KS && !inside ? v4i{0, 0, 0, 0} : bop;
#pragma unroll
        for (int fb = 0; fb < FB; fb++) acc[pb][fb] = P::mfma(a[ks][fb], b, acc[pb][fb]);
      }
    }
    auto at_pixel = [&](int pb, uint32_t x) { return (Acc *)(p.out + ((uint64_t(at.img) * p.oh + at.y0 + pb) * p.ow + x) * p.f + f0 + 4 * lg); };
    if (p.whole_lines) {
      // A pixel's 32 filters are a cache line: lanes of pixels 0 .. 7 and 8 .. 15 exchange a block, so that a store is eight whole
      // lines and not sixteen halves, and they go past the caches (32 x 3 -> 96 x 224^2 bf16 7 x 7: 156 us in halves, 148 in
      // lines, 131 in lines past the caches; halves past the caches 197).
      const bool low = li < 8;
      const uint32_t x = at.x0 + (li & 7);
#pragma unroll
      for (int pb = 0; pb < ITEM_H; pb++) {
        const Acc mine = low ? acc[pb][0] : acc[pb][1];
        Acc theirs = low ? acc[pb][1] : acc[pb][0];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const typename P::Element own = theirs[i];
          const int bits = __builtin_bit_cast(int, own), other = __builtin_amdgcn_update_dpp(bits, bits, 0x128, 0xf, 0xf, false);   // row_ror:8
          theirs[i] = __builtin_bit_cast(typename P::Element, other);
        }
        if (at.y0 + pb >= p.oh) continue;
        Acc *d = at_pixel(pb, x) + (low ? 0 : 4), *e = at_pixel(pb, x + 8) + (low ? 0 : 4);
        Acc v = low ? mine : theirs, w = low ? theirs : mine;
        if (x < p.ow) {
          if (p.accum) v += *d;
          MRL_STORE_ONCE(v, d);
        }
        if (x + 8 < p.ow) {
          if (p.accum) w += *e;
          MRL_STORE_ONCE(w, e);
        }
      }
    } else {
      const uint32_t x = at.x0 + li;
#pragma unroll
      for (int pb = 0; pb < ITEM_H; pb++)
        if (at.y0 + pb < p.oh && x < p.ow) {
          Acc *d = at_pixel(pb, x);
#pragma unroll
          for (int fb = 0; fb < FB; fb++)
            if (fb * 16 < int(nf)) {
              Acc v = acc[pb][fb];
              if (p.accum) v += d[4 * fb];
              d[4 * fb] = v;
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// The same over strips of `strip` output rows: a strip's patch is in LDS at once, where every two rows of the form above fetch theirs with all the rows that
// the windows hang over, and how many rows it has is chosen so that the waves end together (strip_rows).  Two chunks of the next strip's patch are on
// their way under every two rows, into a second patch.  Its start is 0.4 us longer.
template <int KS, int RPS, bool TAIL, int KIND, bool PIXELS, bool STRIPS>
__global__ __launch_bounds__(64 * WAVES, 4) void k_conv_windows(PixelsArgs p) {
  typedef Pixels<KIND> P;
  typedef typename P::Acc Acc;
  typedef typename P::Raw Raw;
  constexpr bool HALVES = P::HALVES;
  constexpr int PB = P::PB, PER_CHUNK = P::PER_CHUNK, STEPS = KS + TAIL, CHUNKS = 4 / RPS, GROUP = 16 * FB;
  constexpr uint32_t filter_row = STEPS * 64 + 16, patch_w = ITEM_W - 1 + PER_CHUNK * CHUNKS, row_bytes = patch_w * PB;
  constexpr int ROWS = RPS * (STEPS - 1) + ITEM_H;      // patch rows that the operands of two output rows start in
  extern __shared__ __attribute__((aligned(16))) uint8_t pix_lds[];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint8_t *patch = pix_lds + wave * p.patch_bytes, *other = patch + WAVES * p.patch_bytes;   // (the filters are staged where the other patches will be)
  const uint32_t f0 = blockIdx.y * GROUP, nf = min(uint32_t(GROUP), p.f - f0);

  const uint32_t patch_pixels = patch_w * p.patch_h;
  struct Corner { uint32_t img, y0, x0; };
  const uint32_t tiles_x = (p.ow + ITEM_W - 1) / ITEM_W, per_image = p.per_image;
  auto corner_of = [&](uint32_t item) {
    const uint32_t img = p.by_image.div(item), in_img = item - img * per_image, ty = p.by_row.div(in_img);
    return Corner{img, ty * p.strip, (in_img - ty * tiles_x) * ITEM_W};
  };
  // The c-th 64 pixels of a patch (past the image's edge: as above; an image is below 2 GiB, so that a lane's offset is 32 bits).
  auto fetch = [&](const Corner &at, int c, Raw &px) {
    const uint8_t *const image = p.image + uint64_t(at.img) * p.image_bytes;
    const uint32_t odd = uint32_t(reinterpret_cast<uintptr_t>(image)) & 3;
    const uint32_t i = lane + c * 64, r = i / patch_w;
    if (i >= patch_pixels) return;
    const uint32_t off = (min(at.y0 + r, p.h - 1) * p.w + min(at.x0 + (i - r * patch_w), p.w - 1)) * p.pixel_bytes + odd;
    px.shift = off & 3;
    const uint32_t *from = reinterpret_cast<const uint32_t *>(image - odd + (off & ~3u));
#pragma unroll
    for (int e = 0; e < P::ES; e++) px.v[e] = from[e];
    px.v[P::ES] = from[px.shift + p.pixel_bytes > 4 * P::ES ? P::ES : P::ES - 1];
  };
  auto put = [&](uint8_t *to, int c, const Raw &px) {
    const uint32_t i = lane + c * 64;
    if (i < patch_pixels) P::put_image(to + i * PB, px, p.pixel_bytes);
  };
  const uint32_t stride = gridDim.x * WAVES;
  uint32_t item = blockIdx.x * WAVES + wave;
  Raw first[STRIP_CHUNKS];   // in flight while the filters are staged
  {
    const Corner at = corner_of(min(item, p.items - 1));
#pragma unroll
    for (int c = 0; c < STRIP_CHUNKS; c++) fetch(at, c, first[c]);
  }
  P::template stage_filters<true>(p, GROUP, f0, nf, filter_row, pix_lds + WAVES * p.patch_bytes);
  v4i a[STEPS][FB];
#pragma unroll
  for (int ks = 0; ks < STEPS; ks++)
#pragma unroll
    for (int fb = 0; fb < FB; fb++) a[ks][fb] = *(const v4i *)(pix_lds + WAVES * p.patch_bytes + (fb * 16 + li) * filter_row + lg * 16 + ks * 64);
  Acc start[FB];   // u8 pixels are multiplied as a - 128: 128 times a filter's sum comes on top
#pragma unroll
  for (int fb = 0; fb < FB; fb++) {
    start[fb] = Acc{};
    if constexpr (KIND == IMG_U8) {
      const v4i ones = v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
      for (int ks = 0; ks < STEPS; ks++) start[fb] = P::mfma(a[ks][fb], ones, start[fb]);
      start[fb] *= 128;
    }
  }
  __syncthreads();   // every wave holds its operands: the other patches may lie there
#pragma unroll
  for (int c = 0; c < STRIP_CHUNKS; c++)
    if (c * 64 < int(patch_pixels)) put(patch, c, first[c]);
  const uint32_t chunk = lg & (CHUNKS - 1), row_of = uint32_t(lg) / CHUNKS;
  const uint32_t in_patch = row_of * row_bytes + li * PB + chunk * 16;
  const uint32_t keep_lo = chunk * PER_CHUNK < p.fw ? 0xffffffffu : 0u, keep_hi = chunk * PER_CHUNK + 1 < p.fw ? 0xffffffffu : 0u;
  const bool inside = KS * RPS + row_of < p.fh;   // of the tail step
  for (; item < p.items; item += stride) {
    const Corner at = corner_of(item);
    const bool more = item + stride < p.items;
    const Corner next = corner_of(more ? item + stride : item);
    // The wave's LDS accesses complete in order: what is left is that the compiler keeps them so.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint32_t end = min(p.oh, at.y0 + p.strip);
    const uint8_t *operands = patch + in_patch;
    int chunks = more ? 0 : STRIP_CHUNKS;   // of the next patch that are in LDS
#pragma unroll 1
    for (uint32_t y0 = at.y0; y0 < end; y0 += ITEM_H, operands += ITEM_H * row_bytes) {
      // Two chunks of the next patch are on their way under every two rows.
      Raw px[2];
      const int c0 = chunks;
      if (c0 < STRIP_CHUNKS) fetch(next, c0, px[0]), fetch(next, c0 + 1, px[1]);
      Acc acc[ITEM_H][FB];
#pragma unroll
      for (int pb = 0; pb < ITEM_H; pb++)
#pragma unroll
        for (int fb = 0; fb < FB; fb++) acc[pb][fb] = start[fb];
#pragma unroll
      for (int r = 0; r < ROWS; r++) {
        v4i bop;
        if constexpr (HALVES) {
          const v2u lo = *(const v2u *)(operands + r * row_bytes) & keep_lo, hi = *(const v2u *)(operands + r * row_bytes + 8) & keep_hi;
          bop = v4i{int(lo[0]), int(lo[1]), int(hi[0]), int(hi[1])};
        } else {
          const uint32_t *w = (const uint32_t *)(operands + r * row_bytes);
          bop = v4i{int(w[0]), int(w[1]), int(w[2]), int(w[3])};
        }
#pragma unroll
        for (int ks = 0; ks < STEPS; ks++) {
          const int pb = r - RPS * ks;
          if (pb < 0 || pb >= ITEM_H) continue;
          const v4i b = HALVES && TAIL && ks == KS && !inside ? v4i{0, 0, 0, 0} : bop;
#pragma unroll
          for (int fb = 0; fb < FB; fb++) acc[pb][fb] = P::mfma(a[ks][fb], b, acc[pb][fb]);
        }
      }
      auto at_pixel = [&](int pb, uint32_t x) { return (Acc *)(p.out + ((uint64_t(at.img) * p.oh + y0 + pb) * p.ow + x) * p.f + f0 + 4 * lg); };
      if (p.whole_lines) {
        // A pixel's 32 filters are a cache line: lanes of pixels 0 .. 7 and 8 .. 15 exchange a block, so that a store is eight whole
        // lines and not sixteen halves, and they go past the caches (32 x 3 -> 96 x 224^2 bf16 7 x 7: 156 us in halves, 148 in
        // lines, 131 in lines past the caches; halves past the caches 197).
        const bool low = li < 8;
        const uint32_t x = at.x0 + (li & 7);
#pragma unroll
        for (int pb = 0; pb < ITEM_H; pb++) {
          const Acc mine = low ? acc[pb][0] : acc[pb][1];
          Acc theirs = low ? acc[pb][1] : acc[pb][0];
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const typename P::Element own = theirs[i];
            const int bits = __builtin_bit_cast(int, own), other = __builtin_amdgcn_update_dpp(bits, bits, 0x128, 0xf, 0xf, false);   // row_ror:8
            theirs[i] = __builtin_bit_cast(typename P::Element, other);
          }
          if (y0 + pb >= end) continue;
          Acc *d = at_pixel(pb, x) + (low ? 0 : 4), *e = at_pixel(pb, x + 8) + (low ? 0 : 4);
          Acc v = low ? mine : theirs, w = low ? theirs : mine;
          if (x < p.ow) {
            if (p.accum) v += *d;
            MRL_STORE_ONCE(v, d);
          }
          if (x + 8 < p.ow) {
            if (p.accum) w += *e;
            MRL_STORE_ONCE(w, e);
          }
        }
      } else {
        const uint32_t x = at.x0 + li;
#pragma unroll
        for (int pb = 0; pb < ITEM_H; pb++)
          if (y0 + pb < end && x < p.ow) {
            Acc *d = at_pixel(pb, x);
#pragma unroll
            for (int fb = 0; fb < FB; fb++)
              if (fb * 16 < int(nf)) {
                Acc v = acc[pb][fb];
                if (p.accum) v += d[4 * fb];
                d[4 * fb] = v;
              }
          }
      }
      if (c0 < STRIP_CHUNKS) put(other, c0, px[0]), put(other, c0 + 1, px[1]), chunks = c0 + 2;
    }
    for (; chunks * 64 < int(patch_pixels) && chunks < STRIP_CHUNKS; chunks++) {
      Raw px;
      fetch(next, chunks, px);
      put(other, chunks, px);
    }
    uint8_t *const t = patch;
    patch = other, other = t;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

template <int KS, int KIND, bool PIXELS = true>
hipError_t launch(const PixelsArgs &p, dim3 grid, size_t lds, hipStream_t stream) {
  static std::atomic<uint64_t> limit{0};
  if (!plan::recording() && lds > 65536) {
    hipError_t e = raise_lds_limit(limit, (const void *)k_conv_windows<KS, KIND, PIXELS>, int(lds));
    if (e != hipSuccess) return e;
  }
  MRL_LAUNCH((k_conv_windows<KS, KIND, PIXELS>), grid, dim3(64 * WAVES), lds, stream, p);
  return plan::last_error();
}
template <int KS>
hipError_t launch_ks(const PixelsArgs &p, int kind, dim3 grid, size_t lds, hipStream_t stream) {
  switch (kind) {
    case IMG_I8: return launch<KS, IMG_I8>(p, grid, lds, stream);
    case IMG_U8: return launch<KS, IMG_U8>(p, grid, lds, stream);
    default: return launch<KS, IMG_BF16>(p, grid, lds, stream);
  }
}

// The form with the filters' operands in registers: `rows` filter rows, `rps` of them to a step.
template <int KS, int RPS, bool TAIL, int KIND, bool PIXELS = true, bool STRIPS = true>
hipError_t launch_strips(const PixelsArgs &p, dim3 grid, size_t lds, hipStream_t stream) {
  MRL_LAUNCH((k_conv_windows<KS, RPS, TAIL, KIND, PIXELS, STRIPS>), grid, dim3(64 * WAVES), lds, stream, p);
  return plan::last_error();
}
template <int KS, int RPS, bool TAIL, int KIND, bool PIXELS = true>
hipError_t launch_held(const PixelsArgs &p, dim3 grid, size_t lds, hipStream_t stream) {
  if (p.strip) return launch_strips<KS, RPS, TAIL, KIND>(p, grid, lds, stream);
  MRL_LAUNCH((k_conv_windows<KS, RPS, TAIL, KIND, PIXELS>), grid, dim3(64 * WAVES), lds, stream, p);
  return plan::last_error();
}
template <int RPS, int KIND>
hipError_t launch_rows(const PixelsArgs &p, dim3 grid, size_t lds, hipStream_t stream) {
  switch (p.fh) {
#define MRL_ROWS(N) case N: return launch_held<N / RPS, RPS, N % RPS != 0, KIND>(p, grid, lds, stream);
    MRL_ROWS(1) MRL_ROWS(2) MRL_ROWS(3) MRL_ROWS(4) MRL_ROWS(5) MRL_ROWS(6)
#undef MRL_ROWS
    default: return launch_held<7 / RPS, RPS, 7 % RPS != 0, KIND>(p, grid, lds, stream);
  }
}
// int8 rows of one or two chunks, bf16 ones of two or four.
bool rows_held(const ConvArgs &c, int kind, uint32_t chunks_log2) {
  return c.fh <= 7 && (kind == IMG_BF16 ? chunks_log2 >= 1 : chunks_log2 <= 1);
}

constexpr uint32_t MAX_KS = 7;

uint32_t chunks_log2_of(const ConvArgs &c, int kind) {   // chunks of 16 bytes of a window's row, as 1, 2 or 4
  const uint32_t pixels = kind == IMG_BF16 ? 2 : 4, chunks = (c.fw + pixels - 1) / pixels;
  return chunks <= 1 ? 0 : chunks <= 2 ? 1 : chunks <= 4 ? 2 : 3;
}

// Output rows of a strip, 0: pairs of rows are faster.  A wave's first item waits for its patch and, longer, for the filters; a unit's second
// workgroup adds to that, by their size; and what a round leaves over is a round.  In us, over those that no choice changes: 0.45 a row (an odd one's pair half), more
// beside a second workgroup, 0.4 a round, and the strips' longer start and code 1.  (us, pairs / strips of so many rows: 16 x 3 -> 64 x 109^2 bf16 7 x 7, 6160 pairs on
// 2048 waves, 15.4 / 13.7 (7), 9 x 4 -> 64 x 115^2 12.4 / 10.1, 11 x 3 -> 32 x 82^2 7.0 / 6.5 (3), u8 17 x 3 -> 16 x 151^2 3 x 3 8.1 / 7.3; 14 x 3 -> 64 x 60^2 bf16
// 3 x 3 5.7, strips of four 6.0.)  From five rounds of pairs on these are the better ones (u8 27 x 3 -> 64 x 146^2 5 x 5 31.4, strips of ten 33.1).
uint32_t strip_rows(const ConvArgs &c, uint32_t patch_w, uint32_t steps, uint32_t groups) {
  const uint64_t units = g_compute_units, waves = std::max<uint64_t>(1, 2 * units / groups) * WAVES, across = (c.ow + ITEM_W - 1) / ITEM_W;
  auto strips = [&](uint32_t rows) { return c.b * across * ((c.oh + rows - 1) / rows); };
  if (strips(ITEM_H) > 4 * waves) return 0;
  auto us = [&](uint32_t rows) {
    const uint64_t n = strips(rows), rounds = (n + waves - 1) / waves;
    const double strip = 0.45 * (rows + (rows & 1) * 0.5);
    return (n + WAVES - 1) / WAVES * groups <= units ? strip : 0.6 + 0.16 * steps + (rounds > 1 ? 0.4 * double(rounds) : 0) + 1.35 * double(rounds) * strip;
  };
  uint32_t best = 0;
  double least = us(ITEM_H) - 1.0;
  for (uint32_t rows = 3; rows <= 12 && patch_w * (rows + c.fh - 1) <= STRIP_CHUNKS * 64; rows++)
    if (us(rows) < least) best = rows, least = us(rows);
  return best;
}

}  // namespace

bool conv_pixels_applicable(const ConvArgs &c, int kind) {
  if (kind < 0 || kind > 2 || c.in_planes || c.out_planes || c.c < 3 || c.c > 4 || c.f % 16 != 0) return false;
  const uint32_t log2 = chunks_log2_of(c, kind), es = kind == IMG_BF16 ? 2 : 1;
  if (log2 > 2 || ((uint64_t(c.fh) << log2) + 3) / 4 > MAX_KS) return false;
  const uint64_t items = uint64_t(c.b) * ((c.oh + ITEM_H - 1) / ITEM_H) * ((c.ow + ITEM_W - 1) / ITEM_W);
  return items < (1ull << 30) && (c.f + 31) / 32 < 65535 && (reinterpret_cast<uintptr_t>(c.out) & 15) == 0 &&
         ((reinterpret_cast<uintptr_t>(c.image) | reinterpret_cast<uintptr_t>(c.filters)) & (es - 1)) == 0;
}

hipError_t launch_conv_pixels(const ConvArgs &c, int kind, hipStream_t stream) {
  if (!conv_pixels_applicable(c, kind)) return hipErrorInvalidValue;
  const uint32_t es = kind == IMG_BF16 ? 2 : 1, pb = 4 * es;
  PixelsArgs p;
  p.image = (const uint8_t *)c.image, p.filters = (const uint8_t *)c.filters, p.out = (int32_t *)c.out;
  p.f = c.f, p.oh = c.oh, p.ow = c.ow, p.fh = c.fh, p.fw = c.fw, p.h = c.oh + c.fh - 1, p.w = c.ow + c.fw - 1;
  p.pixel_bytes = c.c * es, p.accum = c.accum;
  p.whole_lines = c.f % 32 == 0 && (reinterpret_cast<uintptr_t>(c.out) & 127) == 0;
  p.chunks_log2 = chunks_log2_of(c, kind);
  const uint32_t rows_per_step = 4u >> p.chunks_log2, whole = c.fh / rows_per_step;
  p.steps = (c.fh + rows_per_step - 1) / rows_per_step;
  p.slots = p.steps * 64 / pb;
  p.patch_w = ITEM_W - 1 + ((16 / pb) << p.chunks_log2), p.patch_h = ITEM_H + c.fh - 1, p.strip = p.per_image = p.image_bytes = 0;
  p.patch_bytes = ((ITEM_H + p.steps * rows_per_step - 1) * p.patch_w * pb + 15) & ~15u;
  const uint32_t tiles_x = (c.ow + ITEM_W - 1) / ITEM_W, per_image = tiles_x * ((c.oh + ITEM_H - 1) / ITEM_H);
  p.items = c.b * per_image;
  p.by_image = FastDiv(per_image), p.by_row = FastDiv(tiles_x), p.by_slots = FastDiv(p.slots), p.by_patch_w = FastDiv(p.patch_w);
  const double pixels = double(c.b) * c.oh * c.ow;
  // (one or two steps under three or four groups of filters, past three rounds of waves: a patch staged once for all of them is
  // the faster one, us, once / per group: 16 x 3 -> 128 x 100^2 3 x 3 16.9 / 19.4, 12 x 4 -> 96 x 134^2 17.7 / 18.5; 17 x 4 -> 96 x 80^2, two and a half rounds, 11.4 / 10.2)
  const uint32_t groups = (c.f + 16 * FB - 1) / (16 * FB);
  const bool shared_patch = p.steps <= 2 && groups > 2 && c.f <= 128 && uint64_t(p.items) * groups > 3 * 2 * uint64_t(g_compute_units) * WAVES;
  if (!shared_patch && rows_held(c, kind, p.chunks_log2) && p.patch_w * p.patch_h <= HELD * 64) {
    p.strip = uint64_t(p.h) * p.w * p.pixel_bytes < (1ull << 31) ? strip_rows(c, p.patch_w, p.steps, groups) : 0;
    if (p.strip) {
      const uint32_t strips = tiles_x * ((c.oh + p.strip - 1) / p.strip);
      p.patch_h = p.strip + c.fh - 1, p.image_bytes = p.h * p.w * p.pixel_bytes;
      p.items = c.b * strips, p.by_image = FastDiv(strips), p.per_image = strips;
      p.patch_bytes = (((p.strip + 1) / ITEM_H * ITEM_H + p.steps * rows_per_step - 1) * p.patch_w * pb + 15) & ~15u;
    }
    const size_t raw = size_t(std::min<uint32_t>(c.f, 16 * FB)) * c.fh * c.fw * p.pixel_bytes + 32;
    const size_t patches = WAVES * size_t(p.patch_bytes), lds = (p.strip ? patches : 0) + std::max(16 * FB * (p.steps * 64 + 16) + raw, patches);
    const uint32_t wgs = std::min<uint32_t>((p.items + WAVES - 1) / WAVES, std::max(1u, 2 * g_compute_units / groups));
    plan::work(plan::UNIT_STREAM, 0, 1.5 * (pixels * c.f * 4 * (c.accum ? 2 : 1) + double(c.b) * p.h * p.w * p.pixel_bytes), 0,
               4000.0 + (700.0 + 100.0 * p.steps) * double((p.items + wgs * WAVES - 1) / (wgs * WAVES)));
    const dim3 grid(wgs, groups);
    if (kind == IMG_BF16) return rows_per_step == 1 ? launch_rows<1, IMG_BF16>(p, grid, lds, stream) : launch_rows<2, IMG_BF16>(p, grid, lds, stream);
    if (kind == IMG_U8) return rows_per_step == 2 ? launch_rows<2, IMG_U8>(p, grid, lds, stream) : launch_rows<4, IMG_U8>(p, grid, lds, stream);
    return rows_per_step == 2 ? launch_rows<2, IMG_I8>(p, grid, lds, stream) : launch_rows<4, IMG_I8>(p, grid, lds, stream);
  }
  // All filters of up to 128 in one workgroup, so that a pixel is staged once; 32 at a time where that
  // would leave compute units without work.
  const uint64_t wanted = (uint64_t(p.items) + WAVES - 1) / WAVES;
  p.group = c.f <= 32 || wanted * 2 <= g_compute_units ? 32 : c.f <= 128 ? (c.f + 31) & ~31u : 64;
  const uint32_t all_groups = (c.f + p.group - 1) / p.group;
  // behind the filters the patches, and before them the filters as they lie in memory (16 bytes more on either side)
  const size_t raw = size_t(std::min(c.f, p.group)) * c.fh * c.fw * p.pixel_bytes + 32;
  const size_t lds = p.group * (p.steps * 64 + 16) + std::max(raw, WAVES * size_t(p.patch_bytes));
  // Two workgroups to a compute unit walk the items, so that the filters are staged once each.
  const uint32_t wgs = std::min<uint32_t>((p.items + WAVES - 1) / WAVES, std::max(1u, 2 * g_compute_units / all_groups));
  plan::work(plan::UNIT_STREAM, 0, 1.5 * (pixels * c.f * 4 * (c.accum ? 2 : 1) + double(c.b) * p.h * p.w * p.pixel_bytes), 0,
             4000.0 + (1000.0 + 200.0 * p.steps) * double((p.items + wgs * WAVES - 1) / (wgs * WAVES)));   // staging the filters; an item
  const dim3 grid(wgs, all_groups);
  switch (whole) {
    case 0: return launch_ks<0>(p, kind, grid, lds, stream);
    case 1: return launch_ks<1>(p, kind, grid, lds, stream);
    case 2: return launch_ks<2>(p, kind, grid, lds, stream);
    case 3: return launch_ks<3>(p, kind, grid, lds, stream);
    case 4: return launch_ks<4>(p, kind, grid, lds, stream);
    case 5: return launch_ks<5>(p, kind, grid, lds, stream);
    case 6: return launch_ks<6>(p, kind, grid, lds, stream);
    default: return launch_ks<7>(p, kind, grid, lds, stream);
  }
}

}  // namespace mrl
