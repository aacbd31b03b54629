"""Few rows against a k-fastest B whose rows start on words, not on 16-byte chunks."""
import numpy as np
import pytest

import morello_amd as M
import orc
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu
KT = M.layout(0, 2, 1)
KINDS = {"u8": ((M.u8, M.i8, M.i32), [0, 1, 5]), "i8": ((M.i8, M.i8, M.i32), [1, 1, 5]),
         "bf16": ((M.bf16, M.bf16, M.f32), [7, 7, 6]), "f32": ((M.f32, M.f32, M.f32), [6, 6, 6])}
GEN = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16, M.f32: synth.normal_f32}


@pytest.mark.parametrize("types", list(KINDS))
@pytest.mark.parametrize("m,k_bytes,n", [
    (1, 8 * 128 + 4, 1100),     # one word behind whole units
    (7, 16 * 128 - 4, 1031),    # one short of them
    (16, 9 * 128 + 60, 1040),
    (30, 10 * 128 + 20, 1037),  # two blocks of rows
    (45, 11 * 128 + 116, 1050),  # four
    (3, 3 * 128 + 12, 1300),    # fewer units than waves
])
@pytest.mark.parametrize("offset", [0, 1])
def test_rows_that_start_on_words(gpu, types, m, k_bytes, n, offset):
    """Whole units and tails of every length in words, at aligned addresses and a word (and, for smaller elements, an element)
    past one; what lies behind a row's end is the next row, or for the last one poison.  Sums of at most 2500 products."""
    dts, codes = KINDS[types]
    size = {M.bf16: 2, M.f32: 4}.get(dts[0], 1)
    k = k_bytes // size
    A, B = GEN[dts[0]](191, 0, (1, m, k)), GEN[dts[1]](191, 1, (1, k, n))
    C = np.zeros((1, m, n), np.int32 if size == 1 else np.float32)
    spec = M.Matmul([1, m, k, n], dts, [None, KT, None])
    assert spec.plan().kernels == ["k_gemm_skinny"]
    stored = np.ascontiguousarray(B.transpose(0, 2, 1))
    want = orc.matmul([1, m, k, n], codes, A, B, C.copy())
    for lead in ([0, 4 // size] if offset == 0 else [1]):
        held = []
        for x in (A, stored):
            poison = {np.uint8: 255, np.int8: 127, np.uint16: 0x7fc0, np.float32: np.nan}[x.dtype.type]
            h = np.full(x.size + lead + 16, poison, x.dtype)
            h[lead:lead + x.size] = x.reshape(-1)
            held.append(M.DeviceBuffer.from_numpy(h))
        out = M.DeviceBuffer.from_numpy(C)
        spec.run_device([held[0].ptr + lead * size, held[1].ptr + lead * size, out.ptr])
        got = out.to_numpy(C.dtype, C.shape)
        if size == 1:
            assert np.array_equal(got, want)
        else:
            assert float(np.abs(got.astype(np.float64) - want).max() / np.abs(want).max()) < 1e-5
        for d in (*held, out):
            d.free()
