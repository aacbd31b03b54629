"""Few rows of A against a k-fastest B, and small Matmuls, on rows of any alignment
(morello_amd/csrc/gemm_skinny.hip) against the oracle.

Sizes around what the kernels count in: 16 rows and columns to a block (one, two or four row blocks,
one or two column blocks a workgroup), 128 bytes of K a wave takes at a time over eight waves, 16-byte
chunks that rows start in or between."""
import numpy as np
import pytest

import morello_amd as M
import orc
from gpu_util import rel_err, run_spec
from morello_amd import synth

pytestmark = pytest.mark.gpu

KINDS = [((M.u8, M.i8, M.i32), [0, 1, 5]), ((M.i8, M.i8, M.i32), [1, 1, 5]), ((M.bf16, M.bf16, M.f32), [7, 7, 6]),
         ((M.f32, M.f32, M.f32), [6, 6, 6])]
GEN = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16, M.f32: synth.uniform_f32}


def check(dts, codes, shape, accum, k_fastest, kernel):
    b, m, k, n = shape
    A, Bm = GEN[dts[0]](77, 0, (b, m, k)), GEN[dts[1]](77, 1, (b, k, n))
    out_np = np.int32 if dts[2] == M.i32 else np.float32
    C0 = synth.uniform_u8(77, 2, (b, m, n)).astype(out_np) if accum else np.full((b, m, n), 7, out_np)
    spec = M.Matmul(list(shape), dts, layouts=[None, M.layout(0, 2, 1) if k_fastest else None, None], accum=accum)
    assert spec.plan().kernels == [kernel], spec.plan()
    got = run_spec(spec, [A, np.ascontiguousarray(Bm.transpose(0, 2, 1)) if k_fastest else Bm, C0])
    want = orc.matmul(list(shape), codes, A, Bm, C0.copy(), accum)
    if dts[2] == M.i32:
        assert np.array_equal(got, want)
    else:
        # f32 sums of up to 2000 products in another order: 2000^0.5 half-ulps of the largest partial sum
        assert rel_err(got, want) < 1e-5


@pytest.mark.parametrize("dts,codes", KINDS)
@pytest.mark.parametrize("shape,accum", [
    ((1, 1, 64, 1030), False),      # half a unit of bytes, two rows of K of 16-bit elements
    ((1, 3, 1039, 1025), True),     # odd rows, a tail of 15 elements, one column past the last block
    ((2, 16, 1024, 520), False),    # whole units, one for each of the eight waves (bytes)
    ((1, 17, 1153, 1100), False),   # two row blocks, the ninth unit and one element
    ((1, 32, 130, 8208), True),     # two column blocks a workgroup
    ((1, 33, 201, 2064), False),    # four row blocks; rows that are not whole chunks: two column blocks
    ((3, 64, 255, 700), True),
])
def test_few_rows_against_a_k_fastest_b(gpu, dts, codes, shape, accum):
    check(dts, codes, shape, accum, True, "k_gemm_skinny")


@pytest.mark.parametrize("dts,codes", KINDS)
@pytest.mark.parametrize("shape,accum", [
    ((1, 32, 259, 10), False), ((1, 1, 67, 1), True), ((1, 16, 65, 16), False), ((1, 17, 513, 33), True),
    ((2, 100, 333, 211), False),    # more than 128 blocks: two row blocks a workgroup
    ((1, 150, 501, 251), True),
])
def test_small_problems_with_a_row_major_b(gpu, dts, codes, shape, accum):
    check(dts, codes, shape, accum, False, "k_gemm_tiny")


@pytest.mark.parametrize("k", [200, 203])
def test_what_lies_behind_a_rows_end_does_not_count(gpu, k):
    """NaN in the next row of A and of B reaches none of this row's sums."""
    A, Bm = synth.normal_bf16(78, 0, (1, 4, k)), synth.normal_bf16(78, 1, (1, 1100, k))
    A[0, 1], Bm[0, 5] = 0x7fc0, 0x7fc0
    spec = M.Matmul([1, 4, k, 1100], (M.bf16, M.bf16, M.f32), layouts=[None, M.layout(0, 2, 1), None])
    got = run_spec(spec, [A, Bm, np.zeros((1, 4, 1100), np.float32)])[0]
    bad = np.zeros((4, 1100), bool)
    bad[1], bad[:, 5] = True, True
    assert np.array_equal(np.isnan(got), bad)
