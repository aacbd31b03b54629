// f32 Matmul through the bf16 matrix cores: every f32 as three bf16 that add up to it exactly.
//
// The f32 MFMA has a sixteenth of the bf16 one's rate.  A value's upper 16 bits are a bf16 (h); what is left has 16 bits, of
// which the rounded upper half (m) and the rest (l) are bf16 too: x = h + m + l without error, m below 2^-7 |x| and l at most 2^-16 |x|, and
//   x y = h h' + (h m' + m h') + (m m' + h l' + l h') + (m l' + l m') + l l', the last at most 2^-32 |x y| and left out:
// eight MFMAs for sixteen k where the f32 form takes eight of twice the time each.  The products but the first are summed on
// their own, 2^-6 of the first and less, so that a sum of one term is rounded as once (within 2^-24 and a sixteenth of that; without m l' + l m', 3 to 18 % faster, 2^-22).
// Waves that share K add up their first products and their others apart, so that a sum of some terms is rounded at its size about as often (1 to 2 % of the time).
// The roundings of a longer sum, one to sixteen terms and not to two, come to less than those of the f32 MFMA: relative error in the norm for 0.5 x normal
// operands, f32 MFMA / this: two values a row 3.1e-8 / 2.6e-8, four 4.0e-8 / 2.6e-8, 16 7.4e-8 / 3.3e-8, K = 226 2.7e-7 / 6.7e-8, 1024 5.7e-7 / 1.3e-7, 1500 6.9e-7 / 1.6e-7.
// (The three parts: G. Henry, P. Tang and A. Heinecke, Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations, 2019.)
//
// Where the parts would not do, the tile is computed again by the f32 MFMA:
//   - an infinity in A or B leaves a NaN (its m is inf - inf), and so does an overflow on the way;
//   - below 2^-110 the lowest bits of a value may lie below 2^-133, the lowest of a bf16 (the MFMA takes and makes denormals): each thread notes whether it cut
//     such bits off, and the largest magnitude of what it cuts up.  K such losses times that magnitude have to be below half of the last bit of every sum
//     of the tile: beside values of ordinary size they are unless those meet nothing but zeros;
//   - sums below 2^-120, whose parts' products are rounded at 2^-149 more often than the f32 MFMA would.
// The second pass stages the values as they are.  (us, nothing of the kind / an infinity in every sixteenth row / -3.4e38 in every row / all of A below
// 2^-119, beside them the f32 MFMA's own kernel: 2048^3 118 / 159 / 150 / 241, 140; 1000^3 22 / 39 / 26 / 39, 25; 512^3 6.8 / 11.3 / 11.3 / 11.3, 11.5.  From memory without staging, and with
// all values past 2^60 counted among these: 2048^3 328, with a k-fastest B 534, 1000^3 126, 512^3 18.)
//
// What bounds it: of large ones the bf16 MFMAs at what the board's power lets them run at (4096^3 in 848 us is 1.30 PFLOP/s of them, the matrix cores busy 72 % of the
// cycles, where bf16 operands reach 1.42); 64-wide tiles as much by the cutting, six and a half vector instructions a value (37 and 41 % of the cycles, a third in waits); blocks of
// 32 x 32 by the chain of a step (14 and 31 %).
//
// Rows start on any element and are read in place.  The first step takes what K has over whole steps, zeros behind it, so that no
// load but its leaves K and none is masked; rows past M and columns past N are the last one again and are not stored.
// Semantics: morello/src/spec.rs:480-485.
#include "gemm_ring.h"

namespace mrl {
namespace {
using gemm::TileWalk;
using gemm::v4i;
using gemm::v8bf;
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float four_on_word __attribute__((ext_vector_type(4), aligned(4)));

struct Parts { v4i h, m, l; };
// What a thread has cut up so far: the largest magnitude; and, in the lower half, bits that no part has.
struct Seen {
  float most = 0.0f;
  uint32_t lost = 0;
};
// Eight values as three chunks of eight bf16.
__device__ inline Parts cut(const float *x, Seen &seen) {
  Parts p;
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; i++) r[i] = x[i] - __uint_as_float(__float_as_uint(x[i]) & 0xffff0000u);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    p.h[i] = int(__builtin_amdgcn_perm(__float_as_uint(x[2 * i + 1]), __float_as_uint(x[2 * i]), 0x07060302));   // the upper halves
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(seen.most) : "v"(x[2 * i]), "v"(x[2 * i + 1]));
  }
#pragma unroll
  for (int i = 0; i < 4; i++) p.m[i] = __builtin_bit_cast(int, __builtin_convertvector((v2f{r[2 * i], r[2 * i + 1]}), v2bf));
#pragma unroll
  for (int i = 0; i < 4; i++) {
    r[2 * i] -= __uint_as_float(uint32_t(p.m[i]) << 16), r[2 * i + 1] -= __uint_as_float(uint32_t(p.m[i]) & 0xffff0000u);
    asm("v_or3_b32 %0, %0, %1, %2" : "+v"(seen.lost) : "v"(r[2 * i]), "v"(r[2 * i + 1]));
    p.l[i] = int(__builtin_amdgcn_perm(__float_as_uint(r[2 * i + 1]), __float_as_uint(r[2 * i]), 0x07060302));
  }
  return p;
}

__device__ inline v16f mfma(v4i a, v4i b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// Operands of one batch entry (or slice of K), in bytes where they are strides.
struct Problem {
  const uint8_t *a, *b;
  float *c;
  int64_t m, n;
  uint32_t lda_b, ldb_b;
  int k;
  __device__ explicit Problem(const GemmArgs &g) {
    a = (const uint8_t *)((const float *)g.a + int64_t(blockIdx.y) * g.sa), b = (const uint8_t *)((const float *)g.b + int64_t(blockIdx.y) * g.sb);
    c = (float *)g.c + int64_t(blockIdx.y) * g.sc;
    m = g.m, n = g.n, lda_b = uint32_t(g.lda) * 4, ldb_b = uint32_t(g.ldb) * 4;
    k = g.k_total != 0 ? int(min(g.k, g.k_total - blockIdx.y * g.k)) : int(g.k);
  }
};

// Whether a tile's parts did, of the workgroup: `sum`, this thread's of `k` terms, holds nothing infinite, no NaN and no sum below 2^-120 but zeros; and
// what the threads lost counts for nothing in any of them.  (A loss is below 2^-133, so that of a product's two values below 2^-132 times the largest.)
template <int N>
__device__ inline bool parts_did(const Seen &seen, const float (&sum)[N], int k, uint32_t *largest) {
  float probe = 0.0f;
  uint32_t least = ~0u;   // twice the smallest magnitude's bits less one, zeros left out
#pragma unroll
  for (int e = 0; e < N; e++) probe = __builtin_fmaf(0.0f, sum[e], probe), least = min(least, 2 * __float_as_uint(sum[e]) - 1);
  const bool never = probe != probe || least < 2 * __float_as_uint(0x1p-120f) - 1, lost = (seen.lost & 0xffff) != 0;
  if (!__syncthreads_or(never || lost)) return true;
  // (nothing large and no small result, as it mostly is: two barriers, not the largest magnitude's five)
  bool small = seen.most > 0x1p20f;
#pragma unroll
  for (int e = 0; e < N; e++) small = small || !(__builtin_fabsf(sum[e]) >= float(k) * 0x1p-87f);
  if (!__syncthreads_or(never || small)) return true;
  if (__syncthreads_or(never)) return false;
  if (threadIdx.x == 0) *largest = 0;
  __syncthreads();
  atomicMax(largest, __float_as_uint(seen.most));
  __syncthreads();
  const float counts = __uint_as_float(*largest) * (float(k) * 0x1p-107f);
  bool below = false;
#pragma unroll
  for (int e = 0; e < N; e++) below = below || !(__builtin_fabsf(sum[e]) >= counts);
  return !__syncthreads_or(below);
}

// The `share`-th of SHARES parts of a wave's T x T blocks, block after block.  Register i of a block: row 8 (i / 4) + 4 (l / 32) + i % 4, column l % 32.
template <int T, int SHARES>
__device__ inline void store(const Problem &p, int64_t m0, int64_t n0, int share, bool accum, int64_t ldc, const float (&sum)[T * T * 16 / SHARES]) {
  const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
#pragma unroll
  for (int e = 0; e < T * T * 16 / SHARES; e++) {
    const int reg = share * (T * T * 16 / SHARES) + e, block = reg / 16, i = reg % 16;
    const int64_t row = m0 + block / T * 32 + 8 * (i / 4) + 4 * lh + i % 4, col = n0 + block % T * 32 + li;
    if (row < p.m && col < p.n) {
      float *at = p.c + row * ldc + col;
      *at = accum ? sum[e] + *at : sum[e];
    }
  }
}

// The sums of PARTS waves that share T x T blocks meet in LDS, [part][wave of the tile][register][lane]; each wave takes its share.
// `lds`: the first part's, `stride` floats before the next one's, which nobody reads any more once all are here.
template <int T, int PARTS>
__device__ inline void meet(float *lds, int stride, int wave_of_tile, int part, const v16f (&acc)[T][T], float (&sum)[T * T * 16 / PARTS]) {
  constexpr int REGS = T * T * 16, MINE = REGS / PARTS;
  if constexpr (PARTS == 1) {
#pragma unroll
    for (int e = 0; e < REGS; e++) sum[e] = acc[e / 16 / T][e / 16 % T][e % 16];
  } else {
    float *const at = lds + wave_of_tile * (REGS * 64) + (threadIdx.x & 63);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < REGS; e++) at[part * stride + e * 64] = acc[e / 16 / T][e / 16 % T][e % 16];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < MINE; e++) {
      sum[e] = at[(part * MINE + e) * 64];
#pragma unroll
      for (int q = 1; q < PARTS; q++) sum[e] += at[q * stride + (part * MINE + e) * 64];
    }
  }
}

// T x T blocks to a wave, four waves to a tile of 64 T x 64 T; G groups of four waves take every G-th step of 16 k.
template <int T, int G>
struct Staged {
  static constexpr int BM = 64 * T, PART = BM * 32, OPERAND = 3 * PART, STAGE = 2 * OPERAND;
  static constexpr int GROUP = G > 1 && BM * BM * 4 > 2 * STAGE ? BM * BM * 4 : 2 * STAGE;   // a group's two stages, or its sums
};
// A thread cuts eight k of a row of A or a column of B at a time and writes the parts to LDS as the MFMA takes them.  Step j's MFMAs,
// the cutting of step j + 1's values and the loads of step j + 3 run between two barriers, dealt out by the scheduler hints.  Computed again, the same pass
// takes the values to LDS as they are, for the f32 MFMA.
template <int T, int G, bool B_KMAJOR>
__global__ __launch_bounds__(256 * G, T == 2 ? 2 : 4) void k_gemm_f32(MRL_WALK_PARAMS, GemmArgs g) {
  typedef Staged<T, G> S;
  constexpr int BM = S::BM, K = 16;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = wave >> 2, wm = wave >> 1 & 1, wn = wave & 1;
  const int tid = threadIdx.x & 255;
  MRL_WALK_TILE(tile_m, tile_n)
  const int64_t m0 = int64_t(tile_m) * BM, n0 = int64_t(tile_n) * BM;
  const Problem p(g);
  const int steps = (p.k + K - 1) / K, mine = (steps + G - 1) / G, head = p.k - K * (steps - 1);   // (every group passes as many barriers)
  uint8_t *const stages = lds + group * S::GROUP;
  // Where a row's eight k of a half of the lanes lie: the halves change places every four rows, and again every eight, so that neither
  // eight nor sixteen lanes that write both halves of their rows, or read one half of theirs, meet in a bank.
  auto place = [](int row, int half) { return row * 32 + ((half ^ (row >> 2) ^ (row >> 3)) & 1) * 16; };

  // What this thread cuts: of A and of B where T is 2, of A or (waves 2 and 3) of B where it is 1.
  constexpr int OPERANDS = T == 2 ? 2 : 1;
  const uint8_t *from[OPERANDS];
  uint32_t off[OPERANDS];
  int half[OPERANDS], row[OPERANDS], at[OPERANDS];
  int next;   // the step that `from` is at
  const bool second = T == 1 && __builtin_amdgcn_readfirstlane(tid >> 7);   // (a type below, so that no step branches on it)
  auto is_b = [](auto second, int o) { return T == 2 ? o == 1 : decltype(second)::value; };
  auto across = [&](auto second, int o) { return !B_KMAJOR && is_b(second, o); };
  auto begin = [&](auto second) {
    next = min(group, steps - 1);
    asm volatile("" : "+s"(next));   // (or the second pass keeps the first one's addresses, in scratch)
    const int k0 = next == 0 ? 0 : head + K * (next - 1);
#pragma unroll
    for (int o = 0; o < OPERANDS; o++) {
      const int t = T == 2 ? tid : tid & 127;
      row[o] = across(second, o) ? t % BM : t >> 1;
      half[o] = across(second, o) ? __builtin_amdgcn_readfirstlane(t / BM) : t & 1;
      at[o] = (is_b(second, o) ? S::OPERAND : 0) + place(row[o], half[o]);
      if (across(second, o)) {
        from[o] = p.b + n0 * 4 + int64_t(k0 + 8 * half[o]) * p.ldb_b;
        off[o] = uint32_t(min(row[o], int(p.n - n0) - 1)) * 4;
      } else {
        from[o] = (is_b(second, o) ? p.b + n0 * p.ldb_b : p.a + m0 * p.lda_b) + int64_t(k0) * 4;
        off[o] = uint32_t(min(row[o], int((is_b(second, o) ? p.n - n0 : p.m - m0) - 1))) * (is_b(second, o) ? p.ldb_b : p.lda_b) + 32 * half[o];
      }
    }
  };
  Seen seen;

  struct Values { float x[OPERANDS][8]; };
  Values kept[2];
  auto load = [&](auto second, Values &to) {   // this group's next step (past its last: that again)
    const int ahead = next + G >= steps ? 0 : next == 0 ? head + K * (G - 1) : K * G;
#pragma unroll
    for (int o = 0; o < OPERANDS; o++) {
      if (across(second, o)) {
#pragma unroll
        for (int i = 0; i < 8; i++) to.x[o][i] = *(const float *)(from[o] + i * int64_t(p.ldb_b) + off[o]);
        from[o] += ahead * int64_t(p.ldb_b);
      } else {
        const four_on_word lo = *(const four_on_word *)(from[o] + off[o]), hi = *(const four_on_word *)(from[o] + off[o] + 16);
#pragma unroll
        for (int i = 0; i < 4; i++) to.x[o][i] = lo[i], to.x[o][4 + i] = hi[i];
        from[o] += ahead * 4;
      }
    }
    next += ahead ? G : 0;
  };
  auto put = [&](const Values &v, uint8_t *stage) {
#pragma unroll
    for (int o = 0; o < OPERANDS; o++) {
      const Parts c = cut(v.x[o], seen);
      uint8_t *to = stage + at[o];
      *(v4i *)to = c.h, *(v4i *)(to + S::PART) = c.m, *(v4i *)(to + 2 * S::PART) = c.l;
    }
  };

  v16f big[T][T], small[T][T];
#pragma unroll
  for (int r = 0; r < T; r++)
#pragma unroll
    for (int c = 0; c < T; c++)
#pragma unroll
      for (int i = 0; i < 16; i++) big[r][c][i] = small[r][c][i] = 0.0f;
  struct Operands { v4i a[3][T], b[3][T]; };
  const int a_rd = wm * 1024 * T + place(li, lh), b_rd = S::OPERAND + wn * 1024 * T + place(li, lh);
  auto read = [&](const uint8_t *stage, Operands &f) {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int t = 0; t < T; t++) {
        f.a[i][t] = *(const v4i *)(stage + a_rd + i * S::PART + t * 1024);
        f.b[i][t] = *(const v4i *)(stage + b_rd + i * S::PART + t * 1024);
      }
  };
  auto multiply = [&](const Operands &f) {
    auto all = [&](int x, int y, v16f (&acc)[T][T]) {   // (one block after the other: no MFMA waits for the one before it)
#pragma unroll
      for (int r = 0; r < T; r++)
#pragma unroll
        for (int c = 0; c < T; c++) acc[r][c] = mfma(f.a[x][r], f.b[y][c], acc[r][c]);
    };
    all(0, 1, small), all(0, 0, big), all(1, 0, small), all(1, 1, small), all(0, 2, small), all(2, 0, small), all(1, 2, small), all(2, 1, small);
  };
  // The same for the f32 MFMA: 64 bytes of a row, the four chunks of which change places every four rows.
  auto place_f32 = [](int row, int chunk) { return row * 64 + ((chunk ^ (row >> 2)) & 3) * 16; };
  auto put_f32 = [&](auto second, const Values &v, uint8_t *stage) {
#pragma unroll
    for (int o = 0; o < OPERANDS; o++)
#pragma unroll
      for (int q = 0; q < 2; q++)
        *(v4f *)(stage + (is_b(second, o) ? BM * 64 : 0) + place_f32(row[o], 2 * half[o] + q)) = v4f{v.x[o][4 * q], v.x[o][4 * q + 1], v.x[o][4 * q + 2], v.x[o][4 * q + 3]};
  };
  struct OperandsF32 { v4f a[T][2], b[T][2]; };   // lane (l % 32, l / 32): eight k of a row, from 8 (l / 32) on, one to an MFMA
  auto read_f32 = [&](const uint8_t *stage, OperandsF32 &f) {
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        f.a[t][q] = *(const v4f *)(stage + place_f32(32 * (wm * T + t) + li, 2 * lh + q));
        f.b[t][q] = *(const v4f *)(stage + BM * 64 + place_f32(32 * (wn * T + t) + li, 2 * lh + q));
      }
  };
  auto multiply_f32 = [&](const OperandsF32 &f) {
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
      for (int r = 0; r < T; r++)
#pragma unroll
        for (int c = 0; c < T; c++) big[r][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[r][i / 4][i % 4], f.b[c][i / 4][i % 4], big[r][c], 0, 0, 0);
  };
  // All LDS reads and writes are done; loads stay under way.
  auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); };
  // Step j, whose parts (or values) lie in `stage`, while step j + 1's are cut.
  auto step = [&](auto f32, auto second, Values &v, const uint8_t *stage, uint8_t *next_stage) {
    if constexpr (decltype(f32)::value) {
      OperandsF32 f;
      read_f32(stage, f);
      put_f32(second, v, next_stage);
      load(second, v);
      multiply_f32(f);
    } else {
      Operands f;
      read(stage, f);
      put(v, next_stage);
      load(second, v);
      multiply(f);
      __builtin_amdgcn_sched_group_barrier(0x100, 6 * T, 0);   // the reads, then an MFMA and some of the cutting in turn
#pragma unroll
      for (int i = 0; i < 8 * T * T; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, T == 2 ? 4 : 8, 0);
      }
    }
    barrier();
  };
  // False where the parts may not do: a value of this size may make an infinite sum, and so be computed again.  Looked at when 8 steps, 16, 32 and so on are
  // done, so that little is thrown away.  (Not so for rows of tiny values, which a row of probabilities is for most of its way.)
  uint32_t *const given_up = (uint32_t *)(lds + G * S::GROUP);
  auto pass_of = [&](auto f32, auto second) {
    begin(second);
    {
      Values v;
      load(second, v);
      load(second, kept[1]);
      load(second, kept[0]);
      if (group == 0)
#pragma unroll
        for (int o = 0; o < OPERANDS; o++)
#pragma unroll
          for (int i = 0; i < 8; i++)
            if (8 * half[o] + i >= head) v.x[o][i] = 0.0f;
      if constexpr (decltype(f32)::value) put_f32(second, v, stages);
      else put(v, stages);
    }
    if (!decltype(f32)::value && threadIdx.x == 0) *given_up = 0;   // (never while others may be about to read it)
    barrier();
    int j = 0;
    for (int look = decltype(f32)::value ? mine : 8;; look *= 2) {
      for (; j + 2 < min(mine, look); j += 2) {
        step(f32, second, kept[1], stages, stages + S::STAGE);
        step(f32, second, kept[0], stages + S::STAGE, stages);
      }
      if (j + 2 >= mine) break;
      // (read before the next step's barrier, and written again many steps later)
      if (seen.most > 0x1p100f) *given_up = 1;
      barrier();
      if (__builtin_amdgcn_readfirstlane(*given_up)) return false;
    }
    if (j + 1 < mine) step(f32, second, kept[1], stages, stages + S::STAGE);
    if ((mine - 1) * G + group < steps) {   // (behind K's end: nothing)
      const uint8_t *stage = stages + ((mine - 1) & 1) * S::STAGE;
      if constexpr (decltype(f32)::value) {
        OperandsF32 f;
        read_f32(stage, f);
        multiply_f32(f);
      } else {
        Operands f;
        read(stage, f);
        multiply(f);
      }
    }
    return true;
  };
  auto pass = [&](auto f32) { return second ? pass_of(f32, std::true_type{}) : pass_of(f32, std::false_type{}); };

  const int64_t row0 = m0 + wm * 32 * T, col0 = n0 + wn * 32 * T;
  float sum[T * T * 16 / G];
  bool did = pass(std::false_type{});
  if (did) {
    float rest[T * T * 16 / G];
    meet<T, G>((float *)lds, S::GROUP / 4, wave & 3, group, big, sum);
    meet<T, G>((float *)lds, S::GROUP / 4, wave & 3, group, small, rest);
#pragma unroll
    for (int e = 0; e < T * T * 16 / G; e++) sum[e] += rest[e];
    did = parts_did(seen, sum, p.k, (uint32_t *)lds);
  }
  if (!did) {
#pragma unroll
    for (int r = 0; r < T; r++)
#pragma unroll
      for (int c = 0; c < T; c++)
#pragma unroll
        for (int i = 0; i < 16; i++) big[r][c][i] = 0.0f;
    pass(std::true_type{});
    meet<T, G>((float *)lds, S::GROUP / 4, wave & 3, group, big, sum);
  }
  store<T, G>(p, row0, col0, group, g.accum, g.ldc, sum);
}

// A block of 32 x 32 on four waves that take every fourth step of 32 k, operands straight from memory into registers: no barrier and no
// trip through LDS on the way.
constexpr int DEAL = 4;
template <bool B_KMAJOR>
__global__ __launch_bounds__(64 * DEAL, 2) void k_gemm_f32_waves(MRL_WALK_PARAMS, GemmArgs g) {
  constexpr int K = 32, D = 2;
  __shared__ __attribute__((aligned(16))) float part[DEAL * 1024];
  const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  MRL_WALK_TILE(tile_m, tile_n)
  const int64_t m0 = int64_t(tile_m) * 32, n0 = int64_t(tile_n) * 32;
  const Problem p(g);
  const int steps = (p.k + K - 1) / K, head = p.k - K * (steps - 1);
  int next;   // the step that the operands are at
  const uint8_t *a, *b;
  // Lane (l % 32, l / 32): 16 k, from 16 (l / 32) on, of row and column l % 32; eight of them to an MFMA.
  const uint32_t a_off = uint32_t(min(li, int(p.m - m0) - 1)) * p.lda_b + lh * 64, col = uint32_t(min(li, int(p.n - n0) - 1));
  const uint32_t b_off = B_KMAJOR ? col * p.ldb_b + lh * 64 : col * 4 + uint32_t(lh) * 16 * p.ldb_b;
  struct Values { float a[16], b[16]; };
  Values kept[D];
  auto load = [&](Values &v) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const four_on_word x = *(const four_on_word *)(a + a_off + q * 16);
#pragma unroll
      for (int i = 0; i < 4; i++) v.a[q * 4 + i] = x[i];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if constexpr (B_KMAJOR) {
        const four_on_word x = *(const four_on_word *)(b + b_off + q * 16);
#pragma unroll
        for (int i = 0; i < 4; i++) v.b[q * 4 + i] = x[i];
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) v.b[q * 4 + i] = *(const float *)(b + (q * 4 + i) * int64_t(p.ldb_b) + b_off);
      }
    }
    const int ahead = next + DEAL >= steps ? 0 : next == 0 ? head + K * (DEAL - 1) : K * DEAL;   // (past the last: that again)
    a += int64_t(ahead) * 4, b += B_KMAJOR ? int64_t(ahead) * 4 : int64_t(ahead) * p.ldb_b;
    next += ahead ? DEAL : 0;
  };
  Seen seen;
  v16f big[1][1], small[1][1];
#pragma unroll
  for (int i = 0; i < 16; i++) big[0][0][i] = small[0][0][i] = 0.0f;
  auto multiply = [&](const Parts &x, const Parts &y) {
    small[0][0] = mfma(x.h, y.m, small[0][0]);
    big[0][0] = mfma(x.h, y.h, big[0][0]);
    small[0][0] = mfma(x.m, y.h, small[0][0]);
    small[0][0] = mfma(x.m, y.m, small[0][0]);
    small[0][0] = mfma(x.h, y.l, small[0][0]);
    small[0][0] = mfma(x.l, y.h, small[0][0]);
    small[0][0] = mfma(x.m, y.l, small[0][0]);
    small[0][0] = mfma(x.l, y.m, small[0][0]);
  };
  const int mine = steps > wave ? (steps - wave + DEAL - 1) / DEAL : 0;
  auto pass = [&](auto f32) {
    next = min(wave, steps - 1);
    const int k0 = next == 0 ? 0 : head + K * (next - 1);
    a = p.a + m0 * p.lda_b + int64_t(k0) * 4;
    b = B_KMAJOR ? p.b + n0 * p.ldb_b + int64_t(k0) * 4 : p.b + n0 * 4 + int64_t(k0) * p.ldb_b;
    ring::each<D>([&](auto d) { load(kept[decltype(d)::value]); });
    if (wave == 0)
#pragma unroll
      for (int i = 0; i < 16; i++)
        if (16 * lh + i >= head) kept[0].a[i] = kept[0].b[i] = 0.0f;
    for (int left = mine; left > 0;) {
      bool done = false;
      ring::each<D>([&](auto d) {
        Values &v = kept[decltype(d)::value];
        if (!done) {
          if constexpr (decltype(f32)::value) {
#pragma unroll
            for (int i = 0; i < 16; i++) big[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.a[i], v.b[i], big[0][0], 0, 0, 0);
            load(v);
          } else {
            const Parts a0 = cut(v.a, seen), b0 = cut(v.b, seen);
            multiply(a0, b0);
            const Parts a1 = cut(v.a + 8, seen), b1 = cut(v.b + 8, seen);
            load(v);
            multiply(a1, b1);
          }
          done = --left == 0;
        }
      });
    }
  };
  if (mine > 0) pass(std::false_type{});
  float sum[16 / DEAL], rest[16 / DEAL];
  meet<1, DEAL>(part, 1024, 0, wave, big, sum);
  meet<1, DEAL>(part, 1024, 0, wave, small, rest);
#pragma unroll
  for (int e = 0; e < 16 / DEAL; e++) sum[e] += rest[e];
  if (!parts_did(seen, sum, p.k, (uint32_t *)part)) {
#pragma unroll
    for (int i = 0; i < 16; i++) big[0][0][i] = 0.0f;
    if (mine > 0) pass(std::true_type{});
    meet<1, DEAL>(part, 1024, 0, wave, big, sum);
  }
  store<1, DEAL>(p, m0, n0, wave, g.accum, g.ldc, sum);
}

void declare_work(const GemmArgs &g, int side, int k_step, double serial_ns) {
  const double mn = double(g.m) * g.n * g.batch;
  // (1.1 to 1.3 times the rate that the model takes for the f32 MFMA)
  plan::work(plan::UNIT_MFMA_F32, 2.0 * mn * g.k, (double(g.m) * g.k + double(g.k) * g.n) * g.batch * 4 + mn * 4 * (g.accum ? 2 : 1),
             2.0 * side * side * double((g.k + k_step - 1) / k_step * k_step), serial_ns, 1.3);
}

template <int T, int G, bool B_KMAJOR>
hipError_t launch_staged(const GemmArgs &g, hipStream_t stream) {
  typedef Staged<T, G> S;
  constexpr int BM = S::BM, LDS = G * S::GROUP + 16;
  static std::atomic<uint64_t> lds_limit_set{0};
  if (!plan::recording() && LDS > 65536) {
    hipError_t e = raise_lds_limit(lds_limit_set, (const void *)k_gemm_f32<T, G, B_KMAJOR>, LDS);
    if (e != hipSuccess) return e;
  }
  const int tiles_m = int((g.m + BM - 1) / BM), tiles_n = int((g.n + BM - 1) / BM);
  declare_work(g, BM, 16, 2000.0 + (T == 2 ? 700.0 : 400.0) * ((g.k + 15) / 16) / G);
  const TileWalk walk = gemm::tile_walk(tiles_m, tiles_n);
  MRL_LAUNCH((k_gemm_f32<T, G, B_KMAJOR>), dim3(tiles_m * tiles_n, g.batch), dim3(256 * G), LDS, stream, MRL_WALK_ARGS(walk), g);
  return plan::last_error();
}

template <bool B_KMAJOR>
hipError_t launch_waves(const GemmArgs &g, hipStream_t stream) {
  const int tiles_m = int((g.m + 31) / 32), tiles_n = int((g.n + 31) / 32);
  declare_work(g, 32, 32, 2000.0 + 700.0 * ((g.k + 31) / 32) / DEAL);
  const TileWalk walk = gemm::tile_walk(tiles_m, tiles_n);
  MRL_LAUNCH((k_gemm_f32_waves<B_KMAJOR>), dim3(tiles_m * tiles_n, g.batch), dim3(64 * DEAL), 0, stream, MRL_WALK_ARGS(walk), g);
  return plan::last_error();
}

template <int T, int G>
hipError_t launch_either(const GemmArgs &g, hipStream_t stream) {
  return g.b_kmajor ? launch_staged<T, G, true>(g, stream) : launch_staged<T, G, false>(g, stream);
}

}  // namespace

// About `want` slices of K, each of so many; 0: too short for it.  The kernels' first step loads as much of K as any other, in the last slice too: that has
// a step of 32 or more.  (One more step to a slice may leave less than a step again: 1281 in twelve, 128, 160, 192.)
uint32_t gemm_f32_slice_k(uint32_t k, uint32_t want) {
  uint32_t slice_k = (k + want * 32 - 1) / (want * 32) * 32;
  if (slice_k < 128) return 0;
  while (slice_k < k && k % slice_k != 0 && k % slice_k < 32) slice_k += 32;
  return slice_k;
}

// Workgroups of a form go to the compute units in rounds, each as long as a workgroup's steps.  Measured on operands of 1 to 50 MB, B row-major / k-fastest: a
// step of 4 x 32 k of a block of 32 x 32 0.8 / 0.87 us of its unit, however many share it (lines per load, not bytes: the second touches 64 of them), of 2 x 16 k of
// 64 x 64 0.49 / 0.455, of 2 x 16 k of 128 x 128 1.14 / 1.07 to, on all units, 0.4 more; of 16 k of two such workgroups 1.5, of one 0.82; and what a round costs beside its steps.
// Slices of K cost the launch that sums them and their results at 3.1 TB/s.  (us, the f32 MFMA on copies of whole chunks / this, form and slices: 195 x 500 x 621 17.1 / 7.4, waves;
// 192 x 2176 x 128 16.4 / 8.8, waves in 8; twice 382 x 226 x 1179 14.2 / 9.3, 64 wide; 537 x 1668 x 568 23.1 / 17.8, 64 wide in 3; 2048^3 153
// / 122, 128 wide in two groups; 2070 x 389 x 3128 57.7 / 48.6, 128 wide in one; 4096^3 959 / 880.  Over 3100 random sizes 1.35 times as fast, the form chosen within 1.3 % of
// the fastest, geometric means.)
namespace {
enum Form : uint32_t { NONE, WAVES, WIDE_64, WIDE_128, WIDE_128_PAIR };
struct Choice {
  Form form;
  uint32_t slices, slice_k;
  double us;
};
Choice choose(const GemmArgs &g) {
  const double units = g_compute_units;
  const bool nk = g.b_kmajor;
  auto tiles = [&](uint32_t side) { return double((g.m + side - 1) / side) * ((g.n + side - 1) / side) * g.batch; };
  const double t32 = tiles(32), t64 = tiles(64), t128 = tiles(128);
  auto rounds = [&](double n, double at_once) { return double(uint64_t((n + at_once - 1) / at_once)); };
  Choice best{NONE, 1, g.k, 1e300};
  auto consider = [&](Form form, uint32_t slices, uint32_t slice_k, double us) {
    if (us < best.us) best = {form, slices, slice_k, us};
  };
  const double steps = (g.k + 15) / 16, pairs = (g.k + 31) / 32, r128 = rounds(t128, units), r_pair = rounds(t128, 2 * units);
  consider(WIDE_128, 1, g.k, 7.0 + 5.0 * (r128 - 1) + ((nk ? 1.07 : 1.14) + 0.4 * std::min(1.0, t128 / units)) * r128 * pairs);
  consider(WIDE_128_PAIR, 1, g.k, 7.0 + (t128 <= units ? 0.82 * steps : (1.5 * steps + 3.0) * r_pair));
  // (k-fastest rows 512 bytes or a multiple of that apart share the sets of the first cache)
  const double between = nk && g.k % 128 == 0 ? 1.5 : 0.9;
  for (uint32_t want : {1u, 2u, 3u, 4u, 6u, 8u, 12u, 16u}) {
    const uint32_t slice_k = want == 1 ? g.k : gemm_f32_slice_k(g.k, want);
    if (want > 1 && (g.batch != 1 || g.tight || slice_k == 0)) break;
    if (want > 1 && slice_k >= g.k) continue;
    const uint32_t slices = (g.k + slice_k - 1) / slice_k, s32 = (slice_k + 31) / 32;
    const double sum = slices == 1 ? 0.0 : 2.6 + slices * (0.03 + double(g.m) * g.n * 4.0 / 3.1e6);
    const double r32 = rounds(t32 * slices, units), r64 = rounds(t64 * slices, units);
    if (g.k >= 32) consider(WAVES, slices, slice_k, 3.85 + between * (r32 - 1) + (nk ? 0.87 : 0.8) * r32 * ((s32 + DEAL - 1) / DEAL) + sum);
    consider(WIDE_64, slices, slice_k, 4.4 + 1.2 * (r64 - 1) + (nk ? 0.455 : 0.49) * r64 * s32 + sum);
  }
  return best;
}
// k_gemm's 64 x 64 tiles with the f32 MFMA, on rows of whole chunks.
double k_gemm_us(const GemmArgs &g) {
  const double a_unit = double((g.m + 63) / 64) * ((g.n + 63) / 64) * g.batch / g_compute_units, steps = (g.k + 31) / 32;
  return a_unit <= 1 ? 3.4 + 0.68 * steps : a_unit <= 2 ? 4.2 + 1.18 * steps : 5.5 + (0.35 + 0.5 * a_unit) * steps;
}
}  // namespace

// Any rows of f32, from a step of K on.  Whole chunks over a short K, whose start and end are most of the time, stay with k_gemm (640 x 128 x 1632 8.0 us, here
// 8.9, 288 x 128 x 1696 5.6 and 6.3; of a few tiles 160 k and more would gain, 256 x 168 x 768 6.7 and 5.2), and so do those whose tiles its smaller rounds suit better (1472 x
// 256 x 1472 16.8, here 18.8, 2304 x 224 x 2048 25.4 and 27.3, 2 x 576 x 320 x 2176 19.8 and 21.9).
bool gemm_f32_applicable(const GemmArgs &g, int kind) {
  auto words = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 4 == 0; };
  if (kind != 3 || g.k < 16 || !gemm::edge_addressable(g, 4) || g.batch > 65535 || !words(g.a) || !words(g.b) || !words(g.c)) return false;
  if (!gemm_pays(g, kind) || gemv_applicable(g, kind)) return false;
  const bool chunks = g.lda % 4 == 0 && g.ldb % 4 == 0 && g.sa % 4 == 0 && g.sb % 4 == 0 &&
                      reinterpret_cast<uintptr_t>(g.a) % 16 == 0 && reinterpret_cast<uintptr_t>(g.b) % 16 == 0;
  uint32_t left = 0;
  return !chunks || (g.k > 192 && (gemm_tile_side(g, kind) != 64 || gemm_k_splits(g, kind, &left) != 1 || k_gemm_us(g) >= 1.05 * choose(g).us));
}

uint32_t gemm_f32_slices(const GemmArgs &g, uint32_t *slice_k) {
  const Choice c = choose(g);
  *slice_k = c.slice_k;
  return c.slices;
}

hipError_t launch_gemm_f32(const GemmArgs &g, hipStream_t stream) {
  GemmArgs whole = g;
  if (g.k_total != 0) whole.batch = 1, whole.k = g.k_total;   // the form goes by the whole problem
  const Form form = choose(whole).form;
  const uint32_t last = g.k_total != 0 ? g.k_total - (g.batch - 1) * g.k : g.k;
  if (last < (form == WAVES ? 32u : 16u)) return hipErrorInvalidValue;   // (the first step would leave K)
  switch (form) {
    case WAVES: return g.b_kmajor ? launch_waves<true>(g, stream) : launch_waves<false>(g, stream);
    case WIDE_64: return launch_either<1, 2>(g, stream);
    case WIDE_128: return launch_either<2, 2>(g, stream);
    case WIDE_128_PAIR: return launch_either<2, 1>(g, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace mrl
