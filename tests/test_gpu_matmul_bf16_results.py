"""bf16 results of Matmul tiles whose rows start on any element (gemm_ring.h), against float64, with what lies around them."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth

pytestmark = pytest.mark.gpu
KT = M.layout(0, 2, 1)


def _widen(x):
    return (x.astype(np.uint32) << 16).view(np.float32)


# One to sixteen columns over tiles of 64, of 160 (in place) and of 160 behind padded copies; the last tile of a row-major B starts before its neighbour's end.
@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("m,k,n", [(611, 630, 64 * 7 + r) for r in range(1, 17)] + [(2051, 470, 2081), (2040, 470, 2174), (1030, 2310, 4162), (1100, 2310, 4007)])
@pytest.mark.parametrize("at", [0, 1])
def test_rows_of_any_length(gpu, m, k, n, nk, at):
    """Sums of k products in f32 are within k rounding errors of 2^-24 of the sum of magnitudes, and rounded once; what
    lies before and behind the result (`at` elements into its buffer) stays."""
    A, B = synth.normal_bf16(191, 0, (1, m, k)), synth.normal_bf16(191, 1, (1, k, n))
    spec = M.Matmul([1, m, k, n], (M.bf16, M.bf16, M.bf16), [None, KT if nk else None, None])
    assert "k_gemm_ring" in spec.plan().kernels
    guard = 64
    before = np.arange(1, guard + m * n + guard + 1, dtype=np.uint32).astype(np.uint16)
    dA, dB = M.DeviceBuffer.from_numpy(A), M.DeviceBuffer.from_numpy(np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B)
    dC = M.DeviceBuffer.from_numpy(before)
    spec.run_device([dA.ptr, dB.ptr, dC.ptr + 2 * (guard - at)])
    after = dC.to_numpy(np.uint16, before.shape)
    first, end = guard - at, guard - at + m * n
    assert np.array_equal(after[:first], before[:first]) and np.array_equal(after[end:], before[end:])
    a64, b64 = _widen(A[0]).astype(np.float64), _widen(B[0]).astype(np.float64)
    want = a64 @ b64
    bound = (k + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)) + 2.0 ** -8 * np.abs(want)
    assert (np.abs(_widen(after[first:end]).reshape(m, n) - want) <= bound).all()
