"""Middling Matmuls on tiles of 128 rows by 64 to 192 columns (gemm_ring.hip) against float64."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu
KT = M.layout(0, 2, 1)
TYPES = {"u8": (M.u8, M.i8, M.i32), "i8": (M.i8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.f32), "bf16_out": (M.bf16, M.bf16, M.bf16)}


def _widen(x):
    return (x.astype(np.uint32) << 16).view(np.float32) if x.dtype == np.uint16 else x


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("types", ["u8", "i8", "bf16", "bf16_out"])
@pytest.mark.parametrize("b,m,k,n,accum", [
    (1, 1088, 2048, 1024, False),   # 128 x 64 tiles: whole in n, half a tile in m, an even number of steps
    (1, 1025, 2065, 1027, True),    # a row and three columns over, K a byte past whole chunks, an odd number of steps
    (2, 530, 1924, 1100, False),    # two at once
    (1, 1001, 2050, 4425, False),   # 160 columns: the last tile 105 wide
    (1, 2048, 2192, 2560, True),    # whole tiles of 160
    (1, 1793, 1999, 3009, False),   # 192 columns: a row over, the last tile 129 wide
    (1, 1930, 4111, 1922, True),    # bf16: 128 columns
    (2, 1153, 4096, 897, False),
])
def test_middling_matmul(gpu, b, m, k, n, accum, types, nk):
    """Integers exact.  bf16: sums of k products in f32 are within k rounding errors of 2^-24 of the sum of magnitudes,
    in any order; measured against that, far looser than what is seen, and to 1e-6 in the 2-norm.  A bf16 result
    is that rounded once."""
    dts = TYPES[types]
    gen = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16}
    A, B = gen[dts[0]](171, 0, (b, m, k)), gen[dts[1]](171, 1, (b, k, n))
    C = {M.i32: lambda: synth.uniform_i8(171, 2, (b, m, n)).astype(np.int32) * 1001,
         M.f32: lambda: synth.normal_f32(171, 2, (b, m, n)), M.bf16: lambda: synth.normal_bf16(171, 2, (b, m, n))}[dts[2]]()
    spec = M.Matmul([b, m, k, n], dts, [None, KT if nk else None, None], accum)
    if dts[0] == M.bf16 or k < 4096:
        assert "k_gemm_ring" in spec.plan().kernels
    stored = np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B
    got = run_spec(spec, [A, stored, C.copy()])
    a64, b64 = _widen(A).astype(np.float64), _widen(B).astype(np.float64)
    want = a64 @ b64 + (_widen(C).astype(np.float64) if accum else 0)
    if dts[2] == M.i32:
        assert np.array_equal(got, want.astype(np.int32))
        return
    diff = np.abs(_widen(got).astype(np.float64) - want)
    bound = (k + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + 8)
    if dts[2] == M.bf16:
        assert (diff <= bound + 2.0 ** -8 * np.abs(want)).all()
    else:
        assert (diff <= bound).all() and np.linalg.norm(diff) <= 1e-6 * np.linalg.norm(want)


def test_nonfinite_operands_stay_in_their_rows_and_columns(gpu):
    """A NaN and infinities beside the end of K, of M and of N reach the rows and columns that hold them only."""
    m, k, n = 1025, 1033, 1027
    A, B = synth.normal_bf16(172, 0, (1, m, k)), synth.normal_bf16(172, 1, (1, k, n))
    A[0, 7, k - 1], A[0, m - 1, 0], B[0, k - 1, n - 1] = 0x7fc0, 0x7f80, 0xff80
    for nk in (False, True):
        spec = M.Matmul([1, m, k, n], TYPES["bf16"], [None, KT if nk else None, None])
        assert "k_gemm_ring" in spec.plan().kernels
        got = run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, np.zeros((1, m, n), np.float32)])
        finite = np.ones((m, n), bool)
        finite[7], finite[m - 1], finite[:, n - 1] = False, False, False
        assert np.array_equal(np.isfinite(got[0]), finite)
