// The fused Matmul -> Softmax -> Matmul of attention.hip with the KEYS dealt to the waves of a workgroup: for few
// query rows (a decoding step) and for problems whose 128-row workgroups would leave most of the chip idle.
//
// k_attn's other form gives a wave 32 queries of a workgroup's 128 and half of the keys, block after block, with two
// barriers each: its time is a serial chain of blocks (~0.5 us per 64 keys), however few queries there are.  Here a
// workgroup owns 16 * QB queries of one batch entry, every one of its W waves takes every W-th block of 32 keys, and
// the W (maximum, denominator, O) triples meet once at the end, in LDS, by SoftmaxDenominatorAndMaxFromParts' formula
// (morello/src/spec.rs:107-132).  The arithmetic of a block is that of the other form: S^T = K.Q^T and O^T += V^T.P^T in
// 16 x 16 blocks of the bf16 MFMA, P rounded to bf16, the denominators from a row of ones, a reference that moves only
// when some score has outgrown it by 2^40.
//
// A wave is alone with its part of LDS (one K tile, one V tile, 16 KiB at D = 128) and passes no barrier in the loop:
// K of its next block is requested as soon as its operands of this one have been read, V likewise, so that one of the two
// is in flight at any time and eight waves keep 64 to 128 KiB of a compute unit's requests under way.
// What bounds it: the stream of K and V where they are large (16 x 1 x 128 against 32768 keys, 268 MB that no cache holds:
// 53.6 us before, 50.7 now, of which the merging launch and its gap are 5 to 6), and otherwise the trip to memory of a round
// of 256 keys (0.9 us at D = 128 from L2): 4 x 1 x 128 against 564 keys 10.1 -> 5.4 us, 16 x 103 x 80 against 767 11.9 -> 6.7,
// 13 x 346 x 80 against 1088 15.4 -> 9.6.
#include <algorithm>

#include "attention.h"

namespace mrl {
namespace attn {
namespace {

constexpr int KEYS = 32;   // keys per block
// Blocks of a wave whose maxima the reference follows (1024 keys a workgroup): the exponential of the largest score so far is then
// exactly 1, and the largest weigh most in the rounding of P to bf16.  Error in the norm, the form of attention.hip / two
// blocks / four: 19 x 64 x 64 against 1372 keys 1.13e-3 / 1.16e-3 / 0.86e-3, 4 x 700 x 32 against 2048 1.23 / 1.27 / 1.08, 22 x 2 x 64 against
// 1938 1.14 / 1.25 / 1.06, 16 x 1 x 128 against 32768 1.26 / 1.40 / 1.11.  With the maxima over lanes exchanged in the vector unit
// (over_lane_groups) and not through LDS four cost no more than two did: 0.96 of the time over 400 shapes.
constexpr int FOLLOWED = 4;

// The largest of a value over the four lane groups, in all of them.
__device__ inline float over_lane_groups(float x) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const unsigned own = __float_as_uint(x);
  const u2 rows = __builtin_amdgcn_permlane16_swap(own, own, false, false);   // groups 0, 0, 2, 2 and 1, 1, 3, 3
  const float pair = fmaxf(__uint_as_float(rows.x), __uint_as_float(rows.y));
  const unsigned both = __float_as_uint(pair);
  const u2 halves = __builtin_amdgcn_permlane32_swap(both, both, false, false);
  return fmaxf(__uint_as_float(halves.x), __uint_as_float(halves.y));
}

template <int D>
struct Tiles {
  static constexpr int ROW = D * 2, CHUNKS = ROW / 16, SLOTS = ROW / 32;
  static constexpr int TILE = KEYS * ROW;                  // one K or V block
  static constexpr int LOADS = TILE / 1024;                // direct-to-LDS instructions of one
  static constexpr int ROWS_PER_LOAD = 1024 / ROW;
  static constexpr int ROWS_PER_LINE = ROW >= 256 ? 1 : 256 / ROW;   // rows per 256-byte line of banks
  __device__ static constexpr int k_swizzle(int row) { return (row / ROWS_PER_LINE) & (CHUNKS - 1); }
  __device__ static constexpr int v_swizzle(int row) { return (row / ROWS_PER_LINE) & (SLOTS - 1); }
  // The waves' tiles; after the loop their O (QB * D / 16 KiB-sized blocks of a wave) and, behind, maxima and denominators.
  static constexpr int lds_bytes(int qb, int waves) {
    const int triples = waves * (qb * D * 64 + qb * 128), tiles = waves * 2 * TILE;
    return triples > tiles ? triples : tiles;
  }
};

// NARROW: rows of Q and K are `k_in` elements, rows of V `n_out` (multiples of eight), zeros behind them up to D.
template <int D, int QB, int W, bool NARROW>
__global__ __launch_bounds__(64 * W) void k_attn(const void *q, const void *kt, const void *v, float *out, uint32_t b, uint32_t m,
                                                 uint32_t n2, uint32_t n_out, uint32_t key_splits, uint32_t k_in, float *partials) {
  typedef Tiles<D> T;
  constexpr int ROW = T::ROW, TILE = T::TILE, LOADS = T::LOADS;
  constexpr int NC = D / 32, NDB = D / 16;   // k steps of S = K.Q, 16-row blocks of O^T
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lgp = lane >> 4;   // position in a block's 16 rows / columns, lane group
  const uint32_t nqb = (m + 16 * QB - 1) / (16 * QB);
  // (all query blocks of a batch entry share its K and V)
  const uint32_t lin = xcd_run(blockIdx.x, nqb * b);
  const int64_t head = lin / nqb;
  const uint32_t q0 = (lin % nqb) * (16 * QB);
  // This workgroup's blocks of keys: the blockIdx.y-th of key_splits equal shares.
  const uint32_t all_blocks = (n2 + KEYS - 1) / KEYS;
  const uint32_t first = uint32_t(uint64_t(all_blocks) * blockIdx.y / key_splits);
  const uint32_t end = uint32_t(uint64_t(all_blocks) * (blockIdx.y + 1) / key_splits);

  const uint32_t k_row = NARROW ? k_in * 2 : ROW, v_row = NARROW ? n_out * 2 : ROW;   // bytes of a row in memory
  const uint8_t *K = (const uint8_t *)kt + head * n2 * k_row, *V = (const uint8_t *)v + head * n2 * v_row;
  // Rows past n2 lie past the resources' ends: zeros.
  const auto k_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(K), 0, int(n2 * k_row), 0x00020000);
  const auto v_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(V), 0, int(n2 * v_row), 0x00020000);
  uint8_t *const k_tile = lds + wave * 2 * TILE, *const v_tile = k_tile + TILE;

  // Q^T operands: block column qb (queries q0 + 16 qb + l % 16), chunk c of d: lane (l % 16, l / 16) holds d = 32 c + 8 (l / 16) .. + 7.
  v4i qf[QB][NC];
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    const uint8_t *Q = (const uint8_t *)q + (head * m + min(q0 + 16 * qb + lr, m - 1)) * int64_t(k_row);
#pragma unroll
    for (int c = 0; c < NC; c++) {
      if (NARROW && uint32_t(c * 64 + lgp * 16) >= k_row) qf[qb][c] = v4i{0, 0, 0, 0};
      else qf[qb][c] = *(const v4i *)(Q + c * 64 + lgp * 16);
    }
  }

  // One instruction fills 1 KiB of a tile, lane l its 16-byte slot l; K rows are XOR-swizzled by chunk, V rows by
  // 32-byte slot: each lane fetches the chunk that belongs in its slot.
  uint32_t k_src[LOADS], v_src[LOADS];
  {
    const int ld_row = lane / T::CHUNKS, ld_pc = lane % T::CHUNKS;
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
      const int row = i * T::ROWS_PER_LOAD + ld_row;
      const uint32_t k_at = (ld_pc ^ T::k_swizzle(row)) << 4;
      const uint32_t v_at = (((ld_pc >> 1) ^ T::v_swizzle(row)) << 5) | ((ld_pc & 1) << 4);
      k_src[i] = !NARROW || k_at < k_row ? row * k_row + k_at : OUTSIDE;
      v_src[i] = !NARROW || v_at < v_row ? row * v_row + v_at : OUTSIDE;
    }
  }
  const uint32_t k_dst = lds_address(k_tile), v_dst = lds_address(v_tile);
  auto issue_k = [&](uint32_t block) {
#pragma unroll
    for (int i = 0; i < LOADS; i++) dma16_ordered(k_buf, block * (KEYS * k_row) + k_src[i], k_dst + i * 1024);
  };
  auto issue_v = [&](uint32_t block) {
#pragma unroll
    for (int i = 0; i < LOADS; i++) dma16_ordered(v_buf, block * (KEYS * v_row) + v_src[i], v_dst + i * 1024);
  };

  // O^T: block row db (d = 16 db + 4 (l / 16) + i in register i), block column qb; the denominators likewise.
  v4f o[NDB][QB], den[QB];
  float m_run[QB];
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
    m_run[qb] = NO_REFERENCE;
    den[qb] = v4f{0, 0, 0, 0};
#pragma unroll
    for (int db = 0; db < NDB; db++) o[db][qb] = v4f{0, 0, 0, 0};
  }
  const v4i ones = {0x3f803f80, 0x3f803f80, 0x3f803f80, 0x3f803f80};
  // Lane-dependent parts of the operands' addresses: K row l % 16, chunk 4 c + l / 16; V rows 4 (l / 16) .. + 3, slot db.
  uint32_t k_lane[NC], v_lane[NDB];
#pragma unroll
  for (int c = 0; c < NC; c++) k_lane[c] = lr * ROW + (((4 * c + lgp) ^ T::k_swizzle(lr)) << 4);
  {
    const int vrow = 4 * lgp + (lr >> 2);
#pragma unroll
    for (int db = 0; db < NDB; db++) v_lane[db] = vrow * ROW + ((db ^ T::v_swizzle(vrow)) << 5) + (lr & 3) * 8;
  }
  auto mfma = [](v4i a, auto bop, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, bop), c, 0, 0, 0);
  };
  // s_waitcnt vmcnt(LOADS): all but the newest tile's loads.
  constexpr int ALL_BUT_ONE_TILE = 0x0F70 | LOADS, ALL = 0x0F70, READS_DONE = 0xC07F;
  static_assert(LOADS < 16, "the low four bits of the count");

  uint32_t block = first + wave;
  if (block < end) {
    issue_k(block);
    issue_v(block);
    bool start = true;
    __builtin_amdgcn_s_waitcnt(ALL);
    for (; block < end; block += W) {
      const bool more = block + W < end;
      // In flight at this point, oldest first: K of this block, V of this block.
      if (!start) __builtin_amdgcn_s_waitcnt(ALL_BUT_ONE_TILE);
      asm volatile("" ::: "memory");
      v4f s[2][QB];
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
#pragma unroll
        for (int qb = 0; qb < QB; qb++) s[kb][qb] = v4f{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < NC; c++) {
          const v4i a = *(const v4i *)(k_tile + k_lane[c] + kb * 16 * ROW);
#pragma unroll
          for (int qb = 0; qb < QB; qb++) s[kb][qb] = mfma(a, qf[qb][c], s[kb][qb]);
        }
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(READS_DONE);   // K's operands are in registers: its tile may be filled again
      if (more) issue_k(block + W);
      const int valid = int(n2) - int(block * KEYS);
      if (valid < KEYS) {   // keys past n2 leave the softmax
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
          for (int qb = 0; qb < QB; qb++)
#pragma unroll
            for (int r = 0; r < 4; r++)
              if (kb * 16 + 4 * lgp + r >= valid) s[kb][qb][r] = -__builtin_inff();
      }
      auto move_reference = [&]() {
#pragma unroll
        for (int qb = 0; qb < QB; qb++) {
          float mx = s[0][qb][0];
#pragma unroll
          for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int r = 0; r < 4; r++) mx = fmaxf(mx, s[kb][qb][r]);
          mx = over_lane_groups(mx);
          const float m_new = fmaxf(m_run[qb], mx);
          const float alpha = __builtin_amdgcn_exp2f((m_run[qb] - m_new) * LOG2E);
          m_run[qb] = m_new;
          den[qb] *= alpha;
#pragma unroll
          for (int db = 0; db < NDB; db++) o[db][qb] *= alpha;
        }
      };
      // Beyond the followed blocks the reference moves where a score has outgrown it.  (Following every block's maximum would halve
      // the error once more and costs a second round of exponentials wherever some query's moves.)
      const bool fresh = block < first + wave + FOLLOWED * W;
      v8bf pb[QB];
      float pmax = 0.0f;
      auto exponentials = [&]() {
#pragma unroll
        for (int qb = 0; qb < QB; qb++) {
          const float neg_m2 = -m_run[qb] * LOG2E;
#pragma unroll
          for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][qb][r], LOG2E, neg_m2));
              pmax = fmaxf(pmax, e);
              pb[qb][kb * 4 + r] = (__bf16)e;
            }
        }
      };
      if (fresh) move_reference();
      exponentials();
      if (!fresh && __any(!(pmax < STALE_REFERENCE))) {
        move_reference();
        exponentials();
      }
      start = false;
      if (more) __builtin_amdgcn_s_waitcnt(ALL_BUT_ONE_TILE);   // V of this block is in; K of the next may still be under way
      else __builtin_amdgcn_s_waitcnt(ALL);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int db = 0; db < NDB; db++) {
        const v2i lo = read_tr16(v_tile + v_lane[db]), hi = read_tr16(v_tile + v_lane[db] + 16 * ROW);
        const v4i a = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int qb = 0; qb < QB; qb++) o[db][qb] = mfma(a, pb[qb], o[db][qb]);
      }
#pragma unroll
      for (int qb = 0; qb < QB; qb++) den[qb] = mfma(ones, pb[qb], den[qb]);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(READS_DONE);
      if (more) issue_v(block + W);
    }
  }

  // The waves' triples meet: quads of O in LDS as [wave][block column, block row][lane], then [wave][block column][max, denominator][query].
  __syncthreads();   // all tiles have been read
  v4f *const quads = (v4f *)lds;
  float *const stats = (float *)(lds + W * QB * D * 64);
#pragma unroll
  for (int qb = 0; qb < QB; qb++) {
#pragma unroll
    for (int db = 0; db < NDB; db++) quads[((wave * QB + qb) * NDB + db) * 64 + lane] = o[db][qb];
    if (lgp == 0) stats[(wave * QB + qb) * 32 + lr] = m_run[qb], stats[(wave * QB + qb) * 32 + 16 + lr] = den[qb][0];
  }
  __syncthreads();
#pragma unroll
  for (int t = wave; t < QB * NDB; t += W) {
    const int qb = t / NDB, db = t % NDB;
    const uint32_t row = q0 + 16 * qb + lr;
    if (row >= m) continue;
    float mm = -3.0e38f, l = 0.0f;
    float w[W];
#pragma unroll
    for (int i = 0; i < W; i++) w[i] = stats[(i * QB + qb) * 32 + lr], mm = fmaxf(mm, w[i]);
    v4f sum = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < W; i++) {
      w[i] = __builtin_amdgcn_exp2f((w[i] - mm) * LOG2E);
      l += stats[(i * QB + qb) * 32 + 16 + lr] * w[i];
      sum += quads[((i * QB + qb) * NDB + db) * 64 + lane] * w[i];
    }
    const uint32_t col = db * 16 + 4 * lgp;
    if (key_splits > 1) {
      // A partial triple, relative to mm: D + 4 floats (O, maximum, denominator), [query][split].
      float *part = partials + ((head * m + row) * int64_t(key_splits) + blockIdx.y) * (D + 4);
      *(v4f *)(part + col) = sum;
      if (db == 0 && lgp == 0) part[D] = mm, part[D + 1] = l;
      continue;
    }
    sum *= 1.0f / l;
    float *orow = out + (head * m + row) * int64_t(n_out);
    if (NARROW || n_out == D) {   // (rows of whole quads)
      if (!NARROW || col < n_out) *(v4f *)(orow + col) = sum;
    } else {   // padded head dim: columns past n_out are dropped
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (col + r < n_out) orow[col + r] = sum[r];
    }
  }
}

template <int D, int QB, int W, bool NARROW>
hipError_t launch_one(const AttnArgs &a, hipStream_t stream) {
  constexpr int LDS = Tiles<D>::lds_bytes(QB, W), BQ = 16 * QB;
  static std::atomic<uint64_t> lds_limit_set{0};
  if (!plan::recording()) {
    hipError_t e = raise_lds_limit(lds_limit_set, (const void *)k_attn<D, QB, W, NARROW>, LDS);
    if (e != hipSuccess) return e;
  }
  const dim3 grid(((a.m + BQ - 1) / BQ) * a.b, std::max(1u, a.key_splits));
  const double bytes = double(a.b) * (2.0 * a.m * D + 4.0 * a.n2 * D + 4.0 * a.m * a.n_out) + attn_partial_bytes(a, a.key_splits);
  plan::work(plan::UNIT_MFMA_BF16, 4.0 * a.b * a.m * a.n2 * D, bytes,
             1.5 * 4.0 * BQ * D * (double((a.n2 + KEYS - 1) / KEYS) * KEYS / std::max(1u, a.key_splits)), 2000.0);
  MRL_LAUNCH((k_attn<D, QB, W, NARROW>), grid, dim3(64 * W), LDS, stream, a.q, a.kt, a.v, a.out, a.b, a.m, a.n2, a.n_out,
             std::max(1u, a.key_splits), a.k_in, a.partials);
  return plan::last_error();
}

template <int D, int QB>
hipError_t launch_for(const AttnArgs &a, hipStream_t stream) {
  if constexpr (D > 32)
    if (a.k_in) return a.waves == 4 ? launch_one<D, QB, 4, true>(a, stream) : launch_one<D, QB, 8, true>(a, stream);
  return a.waves == 4 ? launch_one<D, QB, 4, false>(a, stream) : launch_one<D, QB, 8, false>(a, stream);
}

}  // namespace
}  // namespace attn

hipError_t launch_attn_keys(const AttnArgs &a, hipStream_t stream) {
  using namespace attn;
  if (a.query_block == 16) {
    switch (a.k) {
      case 32: return launch_for<32, 1>(a, stream);
      case 64: return launch_for<64, 1>(a, stream);
      default: return launch_for<128, 1>(a, stream);
    }
  }
  switch (a.k) {
    case 32: return launch_for<32, 2>(a, stream);
    case 64: return launch_for<64, 2>(a, stream);
    default: return launch_for<128, 2>(a, stream);
  }
}

}  // namespace mrl
