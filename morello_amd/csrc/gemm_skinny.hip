// Matmul with few rows of A against a k-fastest B, and small Matmuls: the matrix cores without the
// tiled kernel's barriers.
//
// The tiled kernel (gemm_mfma_kernel.h) walks K with a barrier and a trip through LDS per 128
// bytes, ~0.45 us each, on four waves, and wants rows that are whole 16-byte chunks.  Here every one of
// a workgroup's eight waves takes its own share of K (units of 128 bytes, dealt round) for the same
// RT x CT blocks of 16 x 16 outputs, waits for nobody on the way, and the waves' partial sums
// meet in LDS once.  Rows may start at any element; those that start on words are read as they lie.
//   semantics: morello/src/spec.rs:480-485; integers exact, bf16 and f32 summed in f32.
#include "gemm_mfma_kernel.h"
#include "row_chunks.h"

namespace mrl {
namespace {
using gemm::v4i;
using gemm::v8bf;
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int WAVES = 8, UNIT = 128;   // bytes of K a wave takes at a time: two MFMA steps

template <int KIND> struct Kind;
template <> struct Kind<0> { typedef v4i Acc; typedef int Out; static constexpr int ES = 1; };
template <> struct Kind<1> : Kind<0> {};
template <> struct Kind<2> { typedef v4f Acc; typedef float Out; static constexpr int ES = 2; };
template <> struct Kind<3> { typedef v4f Acc; typedef float Out; static constexpr int ES = 4; };

// acc += A (16 rows x 64 bytes) . B (64 bytes x 16 columns): lane (l % 16, l / 16) holds the l / 16-th
// 16 bytes of K of row / column l % 16.  Register i of the result: row 4 (l / 16) + i, column l % 16.
template <int KIND>
__device__ inline typename Kind<KIND>::Acc mfma(v4i a, v4i b, typename Kind<KIND>::Acc c) {
  if constexpr (KIND <= 1) return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  else if constexpr (KIND == 2)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  else {
    // four MFMAs of k = 4: the j-th takes the j-th of each lane group's four values from both sides
    const v4f fa = __builtin_bit_cast(v4f, a), fb = __builtin_bit_cast(v4f, b);
#pragma unroll
    for (int j = 0; j < 4; j++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[j], fb[j], c, 0, 0, 0);
    return c;
  }
}

// Sixteen bytes of a row of k_bytes (64 or more), from a multiple of 16 on.  START: what rows start on, K ending on it for 16.
//   4: an access on a word is nearly as fast as one on a chunk (bf16 13 x 2350 x 15509 15.9 us cut out of two chunks, 14.0;
//      30 x 2244 x 7224 13.3, 10.4; u8 25 x 1720 x 5536 8.4, 5.6);
//   1: cut out of the two aligned chunks they lie in: an access that is not on a word runs at a fraction of the
//      rate (u8 4 x 7095 x 6144 14.5 us, cut 11.3), and an aligned chunk that holds a valid byte can be read whole
//      wherever the allocation ends.
typedef int chunk_on_word __attribute__((ext_vector_type(4), aligned(4)));
template <int START>
struct Row {
  typedef v4i Raw;
  const uint8_t *first;
  int k_bytes;
  __device__ void set(const uint8_t *row, int bytes) { first = row, k_bytes = bytes; }
  // all sixteen inside the row
  __device__ Raw fetch(int kb) const {
    if constexpr (START == 16) return *(const v4i *)(first + kb);
    return __builtin_bit_cast(v4i, *(const chunk_on_word *)(first + kb));
  }
  __device__ v4i value(const Raw &r) const { return r; }
  // those behind the row's end are zeros
  __device__ v4i tail(int kb) const {
    const int left = k_bytes - kb;
    if (left <= 0) return v4i{0, 0, 0, 0};
    if constexpr (START == 16) return *(const v4i *)(first + kb);
    // the sixteen that end with the word that holds the row's last byte, and of those the ones asked for
    const int back = left >= 16 ? 0 : (16 - left) & ~3;
    const v4i v = __builtin_bit_cast(v4i, *(const chunk_on_word *)(first + kb - back));
    return left >= 16 ? v : keep_bytes(cut_chunk(v, v4i{0, 0, 0, 0}, uint32_t(back)), left);
  }
};
template <>
struct Row<1> {
  struct Raw { v4i lo, hi; };
  const uint8_t *first;   // the chunk the row's first byte lies in
  int shift;              // where in that chunk
  int k_bytes;
  __device__ void set(const uint8_t *row, int bytes) {
    shift = int(uintptr_t(row) & 15);
    first = row - shift, k_bytes = bytes;
  }
  __device__ Raw fetch(int kb) const {
    Raw r;
    r.lo = *(const v4i *)(first + kb);
    r.hi = *(const v4i *)(first + kb + (shift ? 16 : 0));
    return r;
  }
  __device__ v4i value(const Raw &r) const { return cut_chunk(r.lo, r.hi, uint32_t(shift)); }
  __device__ v4i tail(int kb) const {
    const int left = k_bytes - kb;
    if (left <= 0) return v4i{0, 0, 0, 0};
    Raw r;
    r.lo = *(const v4i *)(first + kb);
    r.hi = *(const v4i *)(first + kb + (shift + min(left, 16) > 16 ? 16 : 0));
    return keep_bytes(value(r), left);
  }
};

// The same of a column of a row-major B, elements ldb_b bytes apart.
template <int ES>
struct Col {
  static constexpr int N = 16 / ES;
  struct Raw { uint32_t e[N]; };
  const uint8_t *first;
  int64_t ldb_b;
  int k;
  __device__ uint32_t at(int kk) const {
    const uint8_t *p = first + int64_t(kk) * ldb_b;
    return ES == 1 ? uint32_t(*p) : ES == 2 ? uint32_t(*(const uint16_t *)p) : *(const uint32_t *)p;
  }
  __device__ Raw fetch(int kb) const {   // (elements behind K repeat the last one)
    Raw r;
#pragma unroll
    for (int i = 0; i < N; i++) r.e[i] = at(min(kb / ES + i, k - 1));
    return r;
  }
  __device__ v4i value(const Raw &r, int kb) const {   // zeros behind K
    v4i v = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < N; i++) v[i * ES / 4] |= int((kb / ES + i < k ? r.e[i] : 0u) << (8 * (i * ES % 4)));
    return v;
  }
};

// The partial sums of the waves into C.  `part`: WAVES x BLOCKS x 256 values of LDS nobody reads any more.
template <int KIND, int RT, int CT>
__device__ inline void finish(const GemmArgs &g, typename Kind<KIND>::Out *part, typename Kind<KIND>::Acc (&acc)[RT][CT],
                              typename Kind<KIND>::Acc (&sums)[CT], int active, int64_t row0, int64_t col0) {
  typedef typename Kind<KIND>::Out Out;
  constexpr int BLOCKS = RT * CT;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int c = 0; c < CT; c++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        Out v = acc[r][c][i];
        // u8 operands were fed as a - 128: 128 times the column sums of B come on top
        if (KIND == 1) v += Out(sums[c][i] * 128);
        part[((wave * BLOCKS + r * CT + c) * 4 + i) * 64 + lane] = v;
      }
  __syncthreads();
  for (int e = threadIdx.x; e < BLOCKS * 256; e += 64 * WAVES) {
    const int blk = e >> 8, i = (e >> 6) & 3, l = e & 63;
    const int64_t row = row0 + (blk / CT) * 16 + (l >> 4) * 4 + i, col = col0 + (blk % CT) * 16 + (l & 15);
    if (row >= int64_t(g.m) || col >= int64_t(g.n)) continue;
    Out sum = part[e];
    for (int w = 1; w < active; w++) sum += part[w * BLOCKS * 256 + e];   // (waves without a share of K wrote zeros)
    const int64_t at = int64_t(blockIdx.z) * g.sc + row * g.ldc + col;
    if (KIND == 2 && g.c_bf16) {
      __bf16 *C = (__bf16 *)g.c;
      if (g.accum) sum += float(C[at]);
      C[at] = __bf16(sum);
    } else {
      Out *C = (Out *)g.c;
      if (g.accum) sum += C[at];
      C[at] = sum;
    }
  }
}

template <int KIND, int RT, int CT>
__device__ inline void multiply(const v4i (&a)[RT], const v4i (&b)[CT], typename Kind<KIND>::Acc (&acc)[RT][CT],
                                typename Kind<KIND>::Acc (&sums)[CT]) {
#pragma unroll
  for (int c = 0; c < CT; c++) {
    if (KIND == 1) sums[c] = mfma<KIND>(v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101}, b[c], sums[c]);
#pragma unroll
    for (int r = 0; r < RT; r++) acc[r][c] = mfma<KIND>(a[r], b[c], acc[r][c]);
  }
}

template <int KIND>
__device__ inline v4i flip(v4i v) {
  if (KIND == 1) v ^= v4i{int(0x80808080), int(0x80808080), int(0x80808080), int(0x80808080)};
  return v;
}

template <int RT, int CT>
constexpr int skinny_lds() {
  return WAVES * (RT + CT) * 16 * UNIT > WAVES * RT * CT * 1024 ? WAVES * (RT + CT) * 16 * UNIT : WAVES * RT * CT * 1024;
}

// B stored k-fastest.  What bounds a large one is the stream over B, and how it is read: eight lanes
// take 128 consecutive bytes of a row, eight rows to a load, and the unit turns into MFMA operands in
// the wave's own 2 KiB of LDS per block (no barrier: nobody else reads it).  Loads straight in the MFMA's form,
// sixteen rows to every sixteen lanes, ask the cache for a line per lane: bf16 64 x 4096 x 4096 25 us that way.
// The next unit is requested as soon as this one has left its registers.
template <int KIND, int START, int RT, int CT>
__global__ __launch_bounds__(64 * WAVES) void k_gemm_skinny(GemmArgs g) {
  typedef typename Kind<KIND>::Acc Acc;
  typedef typename Kind<KIND>::Out Out;
  constexpr int ES = Kind<KIND>::ES, TILES = RT + CT;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row0 = int64_t(blockIdx.y) * (16 * RT), col0 = int64_t(blockIdx.x) * (16 * CT);
  const uint8_t *A = (const uint8_t *)g.a + int64_t(blockIdx.z) * g.sa * ES;
  const uint8_t *B = (const uint8_t *)g.b + int64_t(blockIdx.z) * g.sb * ES;
  const int k_bytes = int(g.k) * ES;
  // Tiles 0 .. RT - 1 are rows of A, the others columns of B; a lane loads the (lane % 8)-th chunk of
  // rows lane / 8 and lane / 8 + 8 of each.  Rows past M and columns past N repeat the last one;
  // their results are not stored.
  const int chunk = lane & 7;
  Row<START> src[TILES][2];
#pragma unroll
  for (int t = 0; t < TILES; t++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int in_tile = (lane >> 3) + 8 * h;
      if (t < RT) src[t][h].set(A + min(row0 + t * 16 + in_tile, int64_t(g.m) - 1) * (g.lda * ES), k_bytes);
      else src[t][h].set(B + min(col0 + (t - RT) * 16 + in_tile, int64_t(g.n) - 1) * (g.ldb * ES), k_bytes);
    }
  uint8_t *patch = lds + wave * (TILES * 16 * UNIT);
  auto put = [&](int t, int h, v4i v) {   // chunks XOR-ed with row / 2: the reads below then spread over the banks
    const int row = (lane >> 3) + 8 * h;
    *(v4i *)(patch + t * (16 * UNIT) + row * UNIT + ((chunk ^ ((row >> 1) & 7)) << 4)) = t < RT ? flip<KIND>(v) : v;
  };
  Acc acc[RT][CT], sums[CT];
#pragma unroll
  for (int c = 0; c < CT; c++) {
    sums[c] = Acc{0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < RT; r++) acc[r][c] = Acc{0, 0, 0, 0};
  }
  auto multiply_patch = [&]() {
    const int row = lane & 15, group = lane >> 4;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      v4i a[RT], b[CT];
#pragma unroll
      for (int t = 0; t < TILES; t++) {
        const v4i v = *(const v4i *)(patch + t * (16 * UNIT) + row * UNIT + (((4 * h + group) ^ ((row >> 1) & 7)) << 4));
        if (t < RT) a[t] = v;
        else b[t - RT] = v;
      }
      multiply<KIND, RT, CT>(a, b, acc, sums);
    }
  };
  const int units = k_bytes / UNIT, rest = k_bytes - units * UNIT;
  typename Row<START>::Raw raw[TILES][2];
  auto fetch = [&](int u) {
#pragma unroll
    for (int t = TILES - 1; t >= 0; t--)
#pragma unroll
      for (int h = 0; h < 2; h++) raw[t][h] = src[t][h].fetch(u * UNIT + chunk * 16);
  };
  int u = wave;
  if (u < units) fetch(u);
  while (u < units) {
#pragma unroll
    for (int t = 0; t < TILES; t++)
#pragma unroll
      for (int h = 0; h < 2; h++) put(t, h, src[t][h].value(raw[t][h]));
    u += WAVES;
    if (u < units) fetch(u);
    __builtin_amdgcn_sched_barrier(0);
    multiply_patch();
  }
  if (rest != 0 && wave == units % WAVES) {
#pragma unroll
    for (int t = 0; t < TILES; t++)
#pragma unroll
      for (int h = 0; h < 2; h++) put(t, h, src[t][h].tail(units * UNIT + chunk * 16));
    multiply_patch();
  }
  __syncthreads();
  finish<KIND, RT, CT>(g, (Out *)lds, acc, sums, min(WAVES, units + (rest != 0 ? 1 : 0)), row0, col0);
}

// B row-major: small problems, whose time is the launch and one round of loads.  Operands come
// straight from memory in the MFMA's form, B's element by element.
template <int KIND, int RT, int CT>
__global__ __launch_bounds__(64 * WAVES) void k_gemm_tiny(GemmArgs g) {
  typedef typename Kind<KIND>::Acc Acc;
  typedef typename Kind<KIND>::Out Out;
  constexpr int ES = Kind<KIND>::ES;
  __shared__ Out part[WAVES * RT * CT * 256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int in16 = lane & 15, group = lane >> 4;
  const int64_t row0 = int64_t(blockIdx.y) * (16 * RT), col0 = int64_t(blockIdx.x) * (16 * CT);
  const uint8_t *A = (const uint8_t *)g.a + int64_t(blockIdx.z) * g.sa * ES;
  const uint8_t *B = (const uint8_t *)g.b + int64_t(blockIdx.z) * g.sb * ES;
  const int k_bytes = int(g.k) * ES;
  Row<1> a_row[RT];
  Col<ES> b_col[CT];
#pragma unroll
  for (int t = 0; t < RT; t++) a_row[t].set(A + min(row0 + t * 16 + in16, int64_t(g.m) - 1) * (g.lda * ES), k_bytes);
#pragma unroll
  for (int t = 0; t < CT; t++) b_col[t] = {B + min(col0 + t * 16 + in16, int64_t(g.n) - 1) * ES, g.ldb * ES, int(g.k)};
  Acc acc[RT][CT], sums[CT];
#pragma unroll
  for (int c = 0; c < CT; c++) {
    sums[c] = Acc{0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < RT; r++) acc[r][c] = Acc{0, 0, 0, 0};
  }
  // steps of 64 bytes, two in flight
  const int steps = (k_bytes + 63) / 64;
  for (int s0 = wave; s0 < steps; s0 += 2 * WAVES) {
    typename Col<ES>::Raw b[2][CT];
    v4i a[2][RT];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int kb = (s0 + i * WAVES) * 64 + group * 16;
#pragma unroll
      for (int c = 0; c < CT; c++) b[i][c] = b_col[c].fetch(kb);
#pragma unroll
      for (int r = 0; r < RT; r++) a[i][r] = a_row[r].tail(kb);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int kb = (s0 + i * WAVES) * 64 + group * 16;
      v4i av[RT], bv[CT];
#pragma unroll
      for (int c = 0; c < CT; c++) bv[c] = b_col[c].value(b[i][c], kb);
#pragma unroll
      for (int r = 0; r < RT; r++) av[r] = flip<KIND>(a[i][r]);
      multiply<KIND, RT, CT>(av, bv, acc, sums);
    }
  }
  finish<KIND, RT, CT>(g, part, acc, sums, min(WAVES, steps), row0, col0);
}

template <int KIND, int RT, int CT>
void declare_work(const GemmArgs &g) {
  constexpr int ES = Kind<KIND>::ES;
  const double mn = double(g.m) * g.n * g.batch;
  plan::work(KIND <= 1 ? plan::UNIT_MFMA_I8 : KIND == 2 ? plan::UNIT_MFMA_BF16 : plan::UNIT_MFMA_F32, 2.0 * mn * g.k,
             (double(g.m) + g.n) * g.k * g.batch * ES + mn * (g.c_bf16 ? 2 : 4) * (g.accum ? 2 : 1), 2.0 * 256 * RT * CT * double(g.k),
             800.0 + 400.0 * double(uint64_t(g.k) * ES / (UNIT * WAVES)));
}

template <int KIND, int START, int RT, int CT>
hipError_t launch_skinny(const GemmArgs &g, hipStream_t stream) {
  constexpr auto kern = k_gemm_skinny<KIND, START, RT, CT>;
  static std::atomic<uint64_t> lds_limit_set{0};
  if (!plan::recording() && skinny_lds<RT, CT>() > 65536) {
    hipError_t e = raise_lds_limit(lds_limit_set, (const void *)kern, skinny_lds<RT, CT>());
    if (e != hipSuccess) return e;
  }
  declare_work<KIND, RT, CT>(g);
  const dim3 grid((g.n + 16 * CT - 1) / (16 * CT), (g.m + 16 * RT - 1) / (16 * RT), g.batch);
  MRL_LAUNCH((k_gemm_skinny<KIND, START, RT, CT>), grid, dim3(64 * WAVES), (skinny_lds<RT, CT>()), stream, g);
  return mrl::plan::last_error();
}

template <int KIND, int START>
hipError_t launch_rows(const GemmArgs &g, hipStream_t stream) {
  // A wider block re-reads A less often (a row block of A is read once per column block); narrower ones
  // give the chip more workgroups.  Up to 16 rows A is no more than B's block: narrow always (bf16
  // 4 x 4096 x 16384 26.4 us, two columns of blocks 34).  Rows that have to be cut out of two chunks are
  // dear on the A side: wide from 128 columns of blocks on (u8 40 x 4001 x 5000 14.1 against 22.4).
  const uint64_t cols = (uint64_t(g.n) + 15) / 16 * g.batch;
  if (g.m <= 16) return launch_skinny<KIND, START, 1, 1>(g, stream);
  if (g.m <= 32) return cols >= 512 ? launch_skinny<KIND, START, 2, 2>(g, stream) : launch_skinny<KIND, START, 2, 1>(g, stream);
  return cols >= (START == 16 ? 512 : 128) ? launch_skinny<KIND, START, 4, 2>(g, stream) : launch_skinny<KIND, START, 4, 1>(g, stream);
}

template <int KIND>
hipError_t launch_kind(const GemmArgs &g, hipStream_t stream) {
  constexpr int ES = Kind<KIND>::ES;
  if (g.b_kmajor) {
    const uintptr_t starts = reinterpret_cast<uintptr_t>(g.a) | uintptr_t(g.lda * ES) | uintptr_t(g.sa * ES) |
                             reinterpret_cast<uintptr_t>(g.b) | uintptr_t(g.ldb * ES) | uintptr_t(g.sb * ES);
    if (starts % 16 == 0 && uint64_t(g.k) * ES % 16 == 0) return launch_rows<KIND, 16>(g, stream);
    // (33 rows and more over up to a unit a wave: cut, us on words / cut: bf16 45 x 398 x 408 5.6 / 5.2, u8 40 x 100 x 2804 twice 5.7 / 4.9;
    // 1336 bytes, 45 x 668 x 325, 7.5 / 7.6)
    if constexpr (ES < 4)
      if (starts % 4 != 0 || (g.m > 32 && uint64_t(g.k) * ES <= UNIT * WAVES)) return launch_rows<KIND, 1>(g, stream);
    return launch_rows<KIND, 4>(g, stream);
  }
  const uint64_t blocks = (uint64_t(g.n) + 15) / 16 * ((uint64_t(g.m) + 15) / 16) * g.batch;
  if (g.m <= 16 || blocks <= 128) {
    declare_work<KIND, 1, 1>(g);
    MRL_LAUNCH((k_gemm_tiny<KIND, 1, 1>), dim3((g.n + 15) / 16, (g.m + 15) / 16, g.batch), dim3(64 * WAVES), 0, stream, g);
  } else {
    declare_work<KIND, 2, 1>(g);
    MRL_LAUNCH((k_gemm_tiny<KIND, 2, 1>), dim3((g.n + 15) / 16, (g.m + 31) / 32, g.batch), dim3(64 * WAVES), 0, stream, g);
  }
  return mrl::plan::last_error();
}

}  // namespace

bool gemm_skinny_applicable(const GemmArgs &g, int kind) {
  const uint64_t es = kind == 3 ? 4 : kind == 2 ? 2 : 1, k_bytes = uint64_t(g.k) * es, b_bytes = k_bytes * g.n * g.batch;
  if (k_bytes < 64 || k_bytes >= (1ull << 31) || g.batch > 65535 || (g.m + 15) / 16 > 65535 || g.n >= (1u << 26)) return false;
  // element-aligned operands
  if (reinterpret_cast<uintptr_t>(g.a) % es || reinterpret_cast<uintptr_t>(g.b) % es) return false;
  const double macs = double(g.m) * g.n * g.k * g.batch;
  const bool chunks = k_bytes % 16 == 0 && g.lda * es % 16 == 0 && g.ldb * es % 16 == 0;
  if (g.b_kmajor) {
    const uint64_t cols = (uint64_t(g.n) + 15) / 16 * g.batch;
    // Few columns and a long K: the tiled kernel with K shared out over workgroups, or, for a row or a few of f32, the dot
    // products.  One workgroup's eight waves take 0.26 us per KB of K (f32 0.4, more rows more), the others 5 to 9 us
    // where K falls into equal slices of rows read in place, and 10 to 20 with their copies or a slice left over (us, this / the
    // others: bf16 1 x 64000 x 14 36.4 / 17.4, 1 x 16000 x 64 10.8 / 5.2, 4 x 10176 x 16 7.7 / 11.9, 10 x 24416 x 16 15.6 / 20.8, 44 x 9600 x 16
    // 15.5 / 7.9; f32 4 x 9792 x 64 16.9 / 7.0).
    if (g.m > 64 || (cols < 64 && macs > 8e6)) return false;
    if (g.batch == 1 && cols < 64 && macs >= 1e5 && k_bytes > 16384) {
      uint32_t left = 0;
      const bool slices = chunks && gemm_k_splits(g, kind, &left) > 1 && left == 0;
      if (g.m > 16 || k_bytes > (slices ? 24576 : 40960)) return false;
    }
    if (kind == 3 && g.batch == 1 && cols < 32 && g.n >= 64 && g.m <= 4 && chunks && k_bytes >= 8192) return false;
    // A short K keeps one to four of the eight waves: past two thousand blocks, which fill the chip several times over, and
    // with columns for more than half of a tile (f32 18643 x (3 x 16 x 16) 36 / 73), the tiled kernel (us, this / that: f32 12 x (53 x 76 x 1533) 18.7 / 7.0, bf16 59 x 64 x 13690 6.3 / 3.0, u8 62 x (3 x 64 x 4096)
    // 22.6 / 10.7; a thousand blocks or 512 bytes are even).
    if (cols * ((g.m + 15) / 16) > 2048 && k_bytes < 512 && g.n > 32) return false;
    if (kind == 3 && g.m > 32 && k_bytes < 256) return false;   // (f32 42 x 22 x 192 4.2 / 2.8)
    // One or two rows against a large B: the dot products (bf16 1 x 2048 x 16384 12.2 us, this 13.3; but
    // 1 x 4096 x 4096 9.5, 8.3).  More than 32 rows of whole chunks: past 8 MB of B the tiled kernel, which reads
    // A less often (bf16 64 x 2048 x 8192 11.5 us, this 12.0; 44 x 1280 x 1265 7.8, 4.9).
    if (gemv_applicable(g, kind) && b_bytes > (40ull << 20)) return false;
    return !(chunks && g.m > 32 && b_bytes > (8ull << 20));
  }
  // Row-major B, a K of a few rounds: small problems (us, padded copies and the tiled kernel / this: bf16
  // 20 x 252 x 75 7.6 / 3.7, f32 32 x 256 x 10 9.9 / 3.7, 251 x 500 x 251 16.1 / 5.8, u8 300^3 8.0 / 4.4), smaller ones where
  // the rows are whole chunks and nothing has to be padded (f32 256^3 7.8 / 4.7, 300 x 100 x 3000 5.9 / 11.8; u8
  // 400^3 4.4 / 6.2; two k steps of the tiled kernel are as short as this).
  // (From sixteen of the tiled kernel's steps on it shares K out over workgroups.)
  // A large C over a short K is stores, which the tiled kernel's larger blocks are better at (f32 794 x 27 x 2728 14.0 us,
  // copies and that one 8.4; 1536 x 16 x 1585 24 / 10); a large B of bytes that needs no copy is read a byte at a time here (u8 21 x
  // (1 x 1891 x 400) 22.2 / 13.7).
  if (k_bytes < 512 && double(g.m) * g.n * g.batch > 4096.0 * double(k_bytes)) return false;
  if (kind <= 1 && g.ldb % 16 == 0 && k_bytes >= 1024 && b_bytes > (4ull << 20)) return false;
  if (k_bytes > 4096 || (k_bytes >= 2048 && macs > 8e6)) return false;
  return chunks ? k_bytes > 256 && macs <= (kind == 3 ? 3e7 : 8e6) : macs <= (kind <= 1 ? 2e7 : 6e7);   // (a byte of B per load)
}

hipError_t launch_gemm_skinny(const GemmArgs &g, int kind, hipStream_t stream) {
  if (!gemm_skinny_applicable(g, kind)) return hipErrorInvalidValue;
  switch (kind) {
    case 0: return launch_kind<0>(g, stream);
    case 1: return launch_kind<1>(g, stream);
    case 2: return launch_kind<2>(g, stream);
    default: return launch_kind<3>(g, stream);
  }
}

}  // namespace mrl
