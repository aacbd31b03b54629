"""f32 Matmuls through the bf16 matrix cores (gemm_f32.hip), against float64."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu
KT = M.layout(0, 2, 1)
F32 = (M.f32,) * 3
FORMS = {"waves": "k_gemm_f32_waves", "64": "k_gemm_f32 [T = 1, G = 2", "128": "k_gemm_f32 [T = 2, G = 2", "pair": "k_gemm_f32 [T = 2, G = 1"}


def _spec(b, m, k, n, nk, accum=False):
    return M.Matmul([b, m, k, n], F32, [None, KT if nk else None, None], accum)


def _run(spec, A, B, C, nk):
    return run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, C.copy()])


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("b,m,k,n,accum,form,slices", [
    (1, 511, 513, 261, False, "waves", 1),    # a step and one k, rows and columns short of a block and one past it
    (1, 331, 385, 501, True, "waves", 1),
    (2, 300, 543, 301, True, "waves", 1),     # 31 k in the first step; two entries
    (1, 33, 4001, 97, False, "waves", 16),    # slices of K, the last one shorter
    (1, 129, 1410, 65, True, "waves", 6),     # ... the old values added in the sum
    (1, 2477, 129, 257, False, "64", 1),      # nine steps on two groups, one k in the first
    (1, 641, 223, 1601, True, "64", 1),
    (3, 130, 175, 1029, True, "64", 1),
    (1, 537, 1667, 569, True, "64", 3),
    (2, 555, 1907, 2969, False, "128", 1),
    (1, 1740, 1751, 1637, True, "128", 1),
    (1, 2071, 389, 3129, True, "pair", 1),
    (1, 1697, 322, 4417, False, "pair", 1),
    (1, 2048, 1024, 2048, False, "128", 1),   # whole tiles, rows of whole chunks
])
def test_f32_matmul_in_parts(gpu, b, m, k, n, accum, form, slices, nk):
    """Within one rounding for every term and those of the parts; and in the norm below 4e-7, where sums
    of two terms at a time come to 3e-7 at K = 500 and 8e-7 at 2048."""
    spec = _spec(b, m, k, n, nk, accum)
    plan = spec.plan()
    assert plan.steps[0].kernel.startswith(FORMS[form]) and plan.kernels[1:] == ["k_sum_splits"] * (slices > 1), plan
    assert plan.steps[0].grid[1] == b * slices
    A, B, C = synth.normal_f32(191, 0, (b, m, k)), synth.normal_f32(191, 1, (b, k, n)), synth.normal_f32(191, 2, (b, m, n))
    got = _run(spec, A, B, C, nk).astype(np.float64)
    a64, b64 = A.astype(np.float64), B.astype(np.float64)
    want = a64 @ b64 + (C if accum else 0)
    assert (np.abs(got - want) <= (k + 4) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + 8)).all()
    assert np.linalg.norm(got - want) <= 4e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("m,k,n", [(511, 513, 261), (2477, 129, 257), (1740, 751, 1637), (2071, 389, 3129), (537, 1667, 569)])
def test_f32_values_that_are_no_three_bf16(gpu, m, k, n, nk):
    """Infinities, the largest finite values, rows and columns of tiny values beside ordinary ones, of zeros, and NaN: as f32
    arithmetic has them, in the tiles that hold them and in the others."""
    A, B = np.abs(synth.normal_f32(192, 0, (1, m, k))), np.abs(synth.normal_f32(192, 1, (1, k, n))) + np.float32(0.01)
    A[0, 3, 7], A[0, 70, k - 1] = np.inf, -np.inf
    A[0, 5] = 0
    A[0, 9] = 0
    A[0, 9, 11] = -3.40282347e38            # the lowest value beside zeros
    B[0, 11] = np.float32(0.5)
    A[0, 100] *= np.float32(1e-36)          # tiny, every one of them: the l and m would be lost
    B[0, :, 20] *= np.float32(1e-35)
    A[0, 130, 2] = np.nan
    want = A[0].astype(np.float64) @ B[0].astype(np.float64)
    spec = _spec(1, m, k, n, nk)
    assert spec.plan().kernels[0].startswith("k_gemm_f32")
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk)[0]
    with np.errstate(over="ignore"):
        want32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want32)) and np.array_equal(np.isinf(got), np.isinf(want32))
    assert np.array_equal(got[np.isinf(got)], want32[np.isinf(want32)])
    normal = np.isfinite(want) & (np.abs(want) >= 2.0 ** -120)   # (below: the products themselves are denormal)
    assert (np.abs(got[normal] - want[normal]) <= 2e-6 * np.abs(want[normal])).all()
    assert normal[100].sum() >= n - 1 and (got[5] == 0).all()


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("m,k,n", [(511, 513, 261), (2477, 129, 257), (1740, 751, 1637), (2071, 389, 3129), (537, 1667, 569)])
def test_f32_tiny_values_that_huge_ones_bring_back(gpu, m, k, n, nk):
    """A tiny value beside a one that meets a zero, times a huge one: the only product of its result, to one rounding."""
    A, B = synth.normal_f32(193, 0, (1, m, k)), synth.normal_f32(193, 1, (1, k, n))
    rows, cols = [50, m - 1], [30, n - 1]
    for i, r in enumerate(rows):
        A[0, r] = 0
        A[0, r, 3], A[0, r, 17] = 1, np.float32(1.2345678e-36) * (i + 1)
    for i, c in enumerate(cols):
        B[0, 3, c], B[0, 17, c] = 0, np.float32(1.7654321e35) * (i + 1)
    spec = _spec(1, m, k, n, nk)
    assert spec.plan().kernels[0].startswith("k_gemm_f32")
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk)[0].astype(np.float64)
    want = A[0].astype(np.float64) @ B[0].astype(np.float64)
    at = np.ix_(rows, cols)
    assert (np.abs(got[at] - want[at]) <= (1 + 2.0 ** -4) * 2.0 ** -24 * np.abs(want[at])).all(), (got[at], want[at])
    assert np.linalg.norm(np.delete(got - want, cols, 1)) <= 4e-7 * np.linalg.norm(np.delete(want, cols, 1))


@pytest.mark.parametrize("m,k,n,nk", [(48, 1281, 1040, False), (272, 1293, 304, True), (400, 1345, 272, False), (112, 1921, 464, False), (144, 2689, 304, True), (112, 3531, 144, False), (720, 3540, 16, True)])
def test_f32_slices_that_nearly_divide_k(gpu, m, k, n, nk):
    """K a little over a number of slices, whose last one was loaded past the operands' ends."""
    spec = _spec(1, m, k, n, nk)
    plan = spec.plan()
    assert plan.kernels == [plan.steps[0].family, "k_sum_splits"] and plan.steps[0].family.startswith("k_gemm_f32"), plan
    A, B = synth.normal_f32(194, 0, (1, m, k)), synth.normal_f32(194, 1, (1, k, n))
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk).astype(np.float64)
    want = A.astype(np.float64) @ B.astype(np.float64)
    assert np.linalg.norm(got - want) <= 4e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("m,k,n,nk,last", [(500, 95, 500, True, 95), (511, 65, 261, True, 65), (300, 47, 301, True, 47), (300, 33, 301, True, 33), (160, 675, 197, False, 35), (157, 689, 194, True, 49)])
def test_f32_tiny_rows_over_fewer_steps_than_waves(gpu, m, k, n, nk, last):
    """A row and a column of nothing but tiny values where some of a tile's waves have no step of K, or of its last slice."""
    A, B = np.abs(synth.normal_f32(195, 0, (1, m, k))), np.abs(synth.normal_f32(195, 1, (1, k, n))) + np.float32(0.01)
    A[0, 100, :k - last] = B[0, :k - last, 20] = 0
    A[0, 100] *= np.float32(1e-36)
    B[0, :, 20] *= np.float32(1e-36)
    spec = _spec(1, m, k, n, nk)
    assert spec.plan().kernels[0] == "k_gemm_f32_waves"
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk)[0].astype(np.float64)
    want = A[0].astype(np.float64) @ B[0].astype(np.float64)
    normal = want >= 2.0 ** -120   # (below: the products themselves are denormal)
    for at in (np.s_[100, :], np.s_[:, 20]):   # (sums of `last` terms)
        assert (np.abs(got - want)[at] <= (last + 4) * 2.0 ** -24 * want[at])[normal[at]].all()
    assert normal[100].sum() >= n - 1 and normal[:, 20].sum() >= m - 1


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("m,k,n", [(511, 513, 261), (2477, 129, 257), (1740, 751, 1637), (2071, 389, 3129), (537, 1667, 569)])
def test_f32_sums_of_one_term_are_rounded_once(gpu, m, k, n, nk):
    """A value a row: each result is one product.  Its parts but for 2^-32 of it, their sum rounded some times at 2^-6 of it and below, and then
    once at its own size: a half of 2^-23 and a sixteenth of that."""
    values, B = synth.normal_f32(196, 0, (m,)), synth.normal_f32(196, 1, (1, k, n))
    A = np.zeros((1, m, k), np.float32)
    at = np.arange(m) * 7 % k
    A[0, np.arange(m), at] = values
    spec = _spec(1, m, k, n, nk)
    assert spec.plan().kernels[0].startswith("k_gemm_f32")
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk)[0].astype(np.float64)
    want = values[:, None].astype(np.float64) * B[0, at].astype(np.float64)
    assert (np.abs(got - want) <= (1 + 2.0 ** -4) * 2.0 ** -24 * np.abs(want)).all()
    assert (got != want.astype(np.float32)).mean() < 0.02   # (near a tie)


def _of_all_sizes(index, shape, lo, hi):
    """Values of magnitudes from 2^lo to 2^hi, all 24 bits of them in use (fewer below 2^-126)."""
    x = synth.normal_f32(197, index, shape)
    mantissa, _ = np.frexp(np.where(x == 0, np.float32(1), x))
    exponents = lo + (np.abs(synth.normal_f32(198, index, shape)) * 1e6).astype(np.int64) % (hi - lo)
    return np.ldexp(mantissa, (exponents + 1).astype(np.int32)).astype(np.float32)


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("m,k", [(511, 501), (2477, 257), (1340, 1637), (6071, 1029), (137, 1667)])
def test_f32_values_down_to_the_smallest_beside_ones(gpu, m, k, nk):
    """Times the identity every value is itself, denormals too, also where a part of it is below the smallest bf16; with a one in every row."""
    A, B = _of_all_sizes(0, (1, m, k), -149, 10), np.eye(k, dtype=np.float32)[None]
    A[0, :, 5] = 1
    spec = _spec(1, m, k, k, nk)
    assert spec.plan().kernels[0].startswith("k_gemm_f32")
    got = _run(spec, A, B, np.zeros((1, m, k), np.float32), nk)
    assert np.array_equal(got, A)


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("lo_a,hi_a,lo_b,hi_b", [(-130, 0, 0, 60), (-70, -50, -80, -50), (-149, 1, -20, 100), (-1, 1, -126, 1), (20, 100, -149, -90)])
@pytest.mark.parametrize("m,k,n", [(511, 513, 261), (2477, 129, 257), (1740, 751, 1637), (2071, 389, 3129), (537, 1667, 569)])
def test_f32_one_term_of_any_size_beside_zeros(gpu, m, k, n, lo_a, hi_a, lo_b, hi_b, nk):
    """A row of A has a one that meets a zero and one value of any size that meets one of any size: the product, rounded once; or, among
    the denormals, within one of the smallest."""
    values, others = _of_all_sizes(1, (m,), lo_a, hi_a), _of_all_sizes(2, (1, k, n), lo_b, hi_b)
    A, B = np.zeros((1, m, k), np.float32), others
    at = 1 + np.arange(m) * 7 % (k - 1)
    A[0, :, 0], B[0, 0] = 1, 0
    A[0, np.arange(m), at] = values
    spec = _spec(1, m, k, n, nk)
    assert spec.plan().kernels[0].startswith("k_gemm_f32")
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk)[0].astype(np.float64)
    want = values[:, None].astype(np.float64) * B[0, at].astype(np.float64)
    assert (np.abs(got - want) <= (1 + 2.0 ** -4) * 2.0 ** -24 * np.abs(want) + np.where(np.abs(want) < 2.0 ** -120, 2.0 ** -149, 0)).all()


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("where", ["early", "late", "last"])
@pytest.mark.parametrize("m,k,n", [(511, 513, 261), (2477, 129, 257), (1740, 1751, 1637), (2071, 389, 3129), (537, 1667, 569)])
def test_f32_values_that_make_infinite_sums(gpu, m, k, n, where, nk):
    """The lowest value once in every third row, met at the start of K, behind its middle or at its end: sums as f32 has them, in the tiles that
    give up on the way and in those that find an infinite one in the end."""
    A, B = synth.normal_f32(199, 0, (1, m, k)), synth.normal_f32(199, 1, (1, k, n))
    rows = np.arange(0, m, 3)
    at = {"early": rows % 11, "late": k // 2 + rows % (k // 2), "last": np.full(rows.size, k - 1)}[where]
    A[0, rows, at] = -3.4e38
    spec = _spec(1, m, k, n, nk)
    assert spec.plan().kernels[0].startswith("k_gemm_f32")
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk)[0].astype(np.float64)
    a64, b64 = A[0].astype(np.float64), B[0].astype(np.float64)
    want, scale = a64 @ b64, np.abs(a64) @ np.abs(b64)
    largest = float(np.finfo(np.float32).max)
    sure = np.abs(np.abs(want) - largest) > 1e-5 * largest
    infinite = sure & (np.abs(want) > largest)
    assert infinite.any() and (got[infinite] == np.sign(want[infinite]) * np.inf).all()
    finite = sure & (np.abs(want) < largest)
    assert (np.abs(got - want)[finite] <= (k + 4) * 2.0 ** -24 * scale[finite]).all()


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("m,k,n", [(511, 513, 261), (2477, 129, 257), (1740, 751, 1637), (2071, 389, 3129)])   # (slices of K round each part of a sum once more, as those of the other kernels do)
def test_f32_sums_of_two_terms(gpu, m, k, n, nk):
    """Two values a row, wherever in K: below 2.9e-8 in the norm, where one rounding of each sum comes to 2.5e-8 (2^-24 over the square root of three, times what a
    significand's distribution makes of it), the f32 MFMA's two to 3.1e-8, and a rounding for every wave that has one of the terms to 3.4e-8."""
    A, B = np.zeros((1, m, k), np.float32), synth.normal_f32(201, 1, (1, k, n))
    rows, first = np.arange(m), np.arange(m) * 13 % k
    A[0, rows, first] = synth.normal_f32(201, 2, (m,))
    A[0, rows, (first + 1 + np.arange(m) * 29 % (k - 1)) % k] = synth.normal_f32(201, 3, (m,))
    spec = _spec(1, m, k, n, nk)
    assert len(spec.plan().kernels) == 1 and spec.plan().kernels[0].startswith("k_gemm_f32")
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk).astype(np.float64)
    want = A.astype(np.float64) @ B.astype(np.float64)
    assert np.linalg.norm(got - want) <= 2.9e-8 * np.linalg.norm(want)


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("m,n", [(2477, 657), (2471, 1257), (3477, 3257)])
@pytest.mark.parametrize("k", [17, 18, 31, 33, 47, 49])
def test_f32_matmul_over_the_fewest_steps(gpu, m, k, n, nk):
    """One to four steps of 16 k on one or two groups of waves, the first of one to sixteen."""
    spec = _spec(1, m, k, n, nk)
    assert spec.plan().kernels == ["k_gemm_f32"]
    A, B = synth.normal_f32(202, 0, (1, m, k)), synth.normal_f32(202, 1, (1, k, n))
    got = _run(spec, A, B, np.zeros((1, m, n), np.float32), nk).astype(np.float64)
    a64, b64 = A.astype(np.float64), B.astype(np.float64)
    assert (np.abs(got - a64 @ b64) <= (k + 4) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))).all()
