// Host check of the copies mrl_run_noalloc chooses (morello_amd/csrc/api.hip): in panels where they fit its fixed scratch, as
// plain rows where only those do, the smallest ones last.  Planning launches nothing.
#include <cstdio>
#include <cstring>

#include "../morello_amd/csrc/kernels.h"

// Bytes of the copies of a bf16 m x k x n with odd rows, K rounded up to whole chunks: A's rows and B's in units of so many
// elements; each starts on 256 bytes.
static uint64_t copies(uint64_t m, uint64_t k, uint64_t n, uint64_t unit_a, uint64_t unit_b, bool whole_k) {
  auto up = [](uint64_t x, uint64_t unit) { return (x + unit - 1) / unit * unit; };
  return up(2 * m * up(k, unit_a), 256) + up(2 * (whole_k ? up(k, 8) : k) * up(n, unit_b), 256);
}

static int check(uint32_t m, uint32_t k, uint32_t n, uint64_t want) {
  mrl_spec spec{};
  spec.kind = MRL_SPEC_MATMUL, spec.rank = 4, spec.n_params = 3;
  spec.spec_shape[0] = 1, spec.spec_shape[1] = m, spec.spec_shape[2] = k, spec.spec_shape[3] = n;
  const uint32_t shapes[3][3] = {{1, m, k}, {1, k, n}, {1, m, n}};
  const int32_t dtypes[3] = {MRL_BF16, MRL_BF16, MRL_F32};
  for (int i = 0; i < 3; i++) spec.dtypes[i] = dtypes[i], mrl_layout_row_major(shapes[i], 3, &spec.layouts[i]);
  mrl_plan plan;
  mrl_plan_step steps[4];
  if (mrl::noalloc_plan(&spec, &plan, steps, 4) != MRL_OK) {
    std::printf("%u x %u x %u: no plan\n", m, k, n);
    return 1;
  }
  if (plan.scratch_bytes == want && plan.n_steps == 2 && std::strstr(steps[1].kernel, "k_gemm_ring")) return 0;
  std::printf("%u x %u x %u: %llu bytes of copies, expected %llu; %s\n", m, k, n, (unsigned long long)plan.scratch_bytes,
              (unsigned long long)want, steps[plan.n_steps - 1].kernel);
  return 1;
}

// i8 with B in strips of 16 columns, which a call lays out as rows: no partial results of slices of K where they do not fit beside them.
static int check_strips(uint32_t m, uint32_t k, uint32_t n) {
  mrl_spec spec{};
  spec.kind = MRL_SPEC_MATMUL, spec.rank = 4, spec.n_params = 3;
  spec.spec_shape[0] = 1, spec.spec_shape[1] = m, spec.spec_shape[2] = k, spec.spec_shape[3] = n;
  const uint32_t a[3] = {1, m, k}, c[3] = {1, m, n};
  spec.dtypes[0] = spec.dtypes[1] = MRL_I8, spec.dtypes[2] = MRL_I32;
  mrl_layout_row_major(a, 3, &spec.layouts[0]), mrl_layout_row_major(c, 3, &spec.layouts[2]);
  const mrl_physdim strips[] = {{2, MRL_DYNAMIC, 0}, {1, MRL_DYNAMIC, 0}, {2, MRL_PACKED, 16}};
  spec.layouts[1].ndims = 3;
  for (int i = 0; i < 3; i++) spec.layouts[1].dims[i] = strips[i];
  mrl_plan usual, plan;
  if (mrl_spec_plan(&spec, &usual, nullptr, 0) != MRL_OK || mrl::noalloc_plan(&spec, &plan, nullptr, 0) != MRL_OK) return std::printf("no plan\n"), 1;
  if (usual.scratch_bytes > MRL_NOALLOC_SCRATCH_BYTES && plan.scratch_bytes <= MRL_NOALLOC_SCRATCH_BYTES) return 0;
  std::printf("i8 %u x %u x %u: %llu bytes, %llu without allocations\n", m, k, n, (unsigned long long)usual.scratch_bytes, (unsigned long long)plan.scratch_bytes);
  return 1;
}

int main() {
  const uint32_t m = 1001, n = 4353;   // tiles of 160 columns
  int bad = check(m, 3041, n, copies(m, 3041, n, 64, 160, true));
  for (uint32_t k : {3061, 3071, 3081}) {   // 33.60 to 33.95 MB in panels, of 33.55; 33.20 to 33.55 as rows
    bad += copies(m, k, n, 64, 160, true) <= MRL_NOALLOC_SCRATCH_BYTES;
    bad += check(m, k, n, copies(m, k, n, 64, 64, true));
  }
  bad += check(m, 3091, n, copies(m, 3091, n, 8, 8, false));
  bad += check_strips(262, 9584, 2896);   // 27.8 MB of rows, 12 of partial results
  if (bad == 0) std::printf("noalloc plans ok\n");
  return bad != 0;
}
