"""The four-wave 256 x 256 tile on ragged shapes and against a k-fastest B (k_gemm_wide with EDGE), against
float64 products: exact for integers (sums stay below 2^53), for bf16 within 1e-5 (f32 sums of up to 6500
products).  33 and more batch entries make the tiles enough for the dispatch to take this one."""
import numpy as np
import pytest

import morello_amd as M
from gpu_util import rel_err, run_spec
from morello_amd import synth

pytestmark = pytest.mark.gpu

KINDS = [(M.u8, M.i8, M.i32), (M.i8, M.i8, M.i32), (M.bf16, M.bf16, M.f32)]


def operands(dts, a_shape, b_shape):
    if dts[0] == M.bf16:
        return synth.normal_bf16(97, 0, a_shape), synth.normal_bf16(97, 1, b_shape)
    gen = synth.uniform_u8 if dts[0] == M.u8 else synth.uniform_i8
    return gen(97, 0, a_shape), synth.uniform_i8(97, 1, b_shape)


def wide(x):
    return (synth.bf16_bits_to_f32(x) if x.dtype == np.uint16 else x).astype(np.float64)


def check(dts, shape, steps, more, accum, k_fastest):
    """K: `steps` times 128 bytes and `more` chunks of 16."""
    b, m, n = shape
    k = (steps * 128 + more * 16) // (2 if dts[0] == M.bf16 else 1)
    A, Bm = operands(dts, (b, m, k), (b, n, k) if k_fastest else (b, k, n))
    np_out = np.float32 if dts[2] == M.f32 else np.int32
    C0 = synth.uniform_i8(97, 2, (b, m, n)).astype(np_out) * (1 if dts[2] == M.f32 else 70001)
    spec = M.Matmul([b, m, k, n], dts, [None, M.layout(0, 2, 1) if k_fastest else None, None], accum)
    assert spec.plan().kernels[-1] == "k_gemm_wide" and "EDGE = true" in spec.plan().steps[-1].kernel, spec.plan()
    got = run_spec(spec, [A, Bm, C0])
    want = np.matmul(wide(A), wide(Bm).transpose(0, 2, 1) if k_fastest else wide(Bm)) + (C0 if accum else 0)
    if dts[2] == M.i32:
        assert np.array_equal(got, want.astype(np.int64).astype(np.int32))
    else:
        assert rel_err(got, want) < 1e-5


# Rows and columns on either side of the waves' halves of a tile; tails of K of none, one and seven chunks;
# step counts odd and even, and those from which an accumulating Spec spaces out its loads of C (26, 98).
@pytest.mark.parametrize("dts", KINDS)
@pytest.mark.parametrize("k_fastest", [False, True])
@pytest.mark.parametrize("shape,steps,more,accum", [
    ((33, 300, 272), 20, 1, False), ((33, 257, 400), 21, 7, False), ((130, 129, 144), 23, 0, False),
    ((33, 384, 512), 20, 0, True), ((33, 270, 496), 24, 7, True), ((33, 300, 272), 26, 3, True), ((33, 257, 272), 99, 1, True),
])
def test_ragged_shapes(gpu, dts, k_fastest, shape, steps, more, accum):
    check(dts, shape, steps, more, accum, k_fastest)


@pytest.mark.parametrize("dts", KINDS)
@pytest.mark.parametrize("steps,accum", [(20, False), (32, True)])
def test_whole_tiles_against_a_k_fastest_b(gpu, dts, steps, accum):
    check(dts, (33, 512, 512), steps, 0, accum, True)


@pytest.mark.parametrize("k_fastest", [False, True])
def test_the_tail_of_k_is_counted_once_whatever_it_holds(gpu, k_fastest):
    """Tile 0 overlaps the last whole one: infinities there must not meet the zeros of the overlap."""
    b, m, n, k = 33, 300, 272, 20 * 64 + 8
    A, Bm = operands((M.bf16,) * 3, (b, m, k), (b, n, k) if k_fastest else (b, k, n))
    A[:, 7, k - 40] = 0x7f80     # +inf, in the overlap of tile 0 and the last whole tile
    spec = M.Matmul([b, m, k, n], (M.bf16, M.bf16, M.f32), [None, M.layout(0, 2, 1) if k_fastest else None, None])
    got = run_spec(spec, [A, Bm, np.zeros((b, m, n), np.float32)])
    row = Bm[:, :, k - 40] if k_fastest else Bm[:, k - 40, :]
    assert np.array_equal(got[:, 7], np.where(synth.bf16_bits_to_f32(row) > 0, np.inf, -np.inf))
    assert np.isfinite(np.delete(got, 7, axis=1)).all()


@pytest.mark.parametrize("k_fastest", [False, True])
@pytest.mark.parametrize("shape,steps,more", [((33, 300, 272), 20, 1), ((33, 257, 401), 21, 7), ((33, 512, 488), 24, 0)])
def test_a_bf16_result_is_the_f32_sum_rounded(gpu, k_fastest, shape, steps, more):
    """The same loop forms both; rows of an odd number of two-byte elements, tiles that end inside a block."""
    b, m, n = shape
    k = (steps * 128 + more * 16) // 2
    A, Bm = operands((M.bf16,) * 3, (b, m, k), (b, n, k) if k_fastest else (b, k, (n + 7) // 8 * 8))
    n = n if k_fastest else Bm.shape[2]
    results = []
    for out, zero in ((M.f32, np.float32), (M.bf16, np.uint16)):
        spec = M.Matmul([b, m, k, n], (M.bf16, M.bf16, out), [None, M.layout(0, 2, 1) if k_fastest else None, None])
        assert spec.plan().kernels[-1] == "k_gemm_wide" and "EDGE = true" in spec.plan().steps[-1].kernel, spec.plan()
        results.append(run_spec(spec, [A, Bm, np.full((b, m, n), 7, zero)]))
    assert np.array_equal(results[1], synth.f32_to_bf16_bits(results[0]))


@pytest.mark.parametrize("dts", KINDS)
@pytest.mark.parametrize("k_fastest", [False, True])
@pytest.mark.parametrize("shape,k_bytes,accum", [((33, 300, 271), 20 * 128 + 6, False), ((33, 257, 403), 24 * 128 - 2, True)])
def test_a_k_of_no_whole_chunks_through_padded_copies(gpu, dts, k_fastest, shape, k_bytes, accum):
    """Copies that hold zeros up to the next chunk of K, rows of them for a row-major B."""
    b, m, n = shape
    k = k_bytes // (2 if dts[0] == M.bf16 else 1)
    A, Bm = operands(dts, (b, m, k), (b, n, k) if k_fastest else (b, k, n))
    C0 = synth.uniform_i8(97, 2, (b, m, n)).astype(np.float32 if dts[2] == M.f32 else np.int32)
    spec = M.Matmul([b, m, k, n], dts, [None, M.layout(0, 2, 1) if k_fastest else None, None], accum)
    assert spec.plan().kernels == ["k_pad_rows_pair", "k_gemm_wide"], spec.plan()
    got = run_spec(spec, [A, Bm, C0])
    want = np.matmul(wide(A), wide(Bm).transpose(0, 2, 1) if k_fastest else wide(Bm)) + (C0 if accum else 0)
    if dts[2] == M.i32:
        assert np.array_equal(got, want.astype(np.int64).astype(np.int32))
    else:
        assert rel_err(got, want) < 1e-5
