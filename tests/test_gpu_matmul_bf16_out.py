"""bf16 Matmuls whose result is bf16: every kernel that stores it rounds the f32 sum (the old value
included) once.  The same kernels form the f32 sums of the f32-output Spec, in the same order, so its
result rounded on the host has to be the bf16 result bit for bit."""
import numpy as np
import pytest

import morello_amd as M
from gpu_util import run_spec
from morello_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [
    (1, 5, 200, 1100), (1, 40, 77, 1030),    # few rows (k-fastest B), small (row-major B)
    (1, 300, 520, 413), (2, 129, 1000, 260),  # 64 tile, ragged and in whole chunks
    (1, 1100, 264, 1300),                     # 128 tile
    (1, 2900, 520, 2100),                     # 256 tile, ragged
    (1, 2560, 256, 2560),                     # 256 tile, whole
    (1, 130, 8256, 70),                       # K in slices
    (1, 1, 2048, 12000),                      # dot products
])
@pytest.mark.parametrize("accum", [False, True])
@pytest.mark.parametrize("k_fastest", [False, True])
def test_bf16_result_is_the_f32_result_rounded(gpu, shape, accum, k_fastest):
    b, m, k, n = shape
    A, Bm = synth.normal_bf16(79, 0, (b, m, k)), synth.normal_bf16(79, 1, (b, n, k) if k_fastest else (b, k, n))
    old = synth.normal_bf16(79, 2, (b, m, n), 8.0) if accum else np.zeros((b, m, n), np.uint16)
    layouts = [None, M.layout(0, 2, 1) if k_fastest else None, None]
    wide = M.Matmul(list(shape), (M.bf16, M.bf16, M.f32), layouts, accum)
    narrow = M.Matmul(list(shape), (M.bf16, M.bf16, M.bf16), layouts, accum)
    want = synth.f32_to_bf16_bits(run_spec(wide, [A, Bm, synth.bf16_bits_to_f32(old)]))
    got = run_spec(narrow, [A, Bm, old.copy()])
    if [s.kernel for s in wide.plan().steps] == [s.kernel for s in narrow.plan().steps]:
        assert np.array_equal(got, want)
    else:
        # another kernel's order of summing (at most 2^-15 of a sum of this size) may tip a tie: a step of bf16
        assert np.abs(got.view(np.int16).astype(np.int32) - want.view(np.int16).astype(np.int32)).max() <= 1


@pytest.mark.parametrize("shape,k_fastest", [
    ((1, 300, 520, 413), False), ((1, 1100, 264, 1300), True), ((1, 2900, 2600, 2100), False),  # 64, 128 and ragged 256 tile
    ((1, 2560, 256, 2560), False), ((1, 2560, 2560, 2560), True),                               # whole 256 tiles
    ((1, 1001, 2050, 4425), False), ((1, 130, 8256, 70), False), ((1, 1, 2048, 12000), True),   # ring, K in slices, dot products
])
@pytest.mark.parametrize("accum", [False, True])
def test_bf16_result_on_any_element(gpu, shape, k_fastest, accum):
    """An output that starts on an odd element goes through the same kernels as an aligned one: the same bits
    (the generic kernel's order of summing gives others)."""
    b, m, k, n = shape
    A, Bm = synth.normal_bf16(80, 0, (b, m, k)), synth.normal_bf16(80, 1, (b, n, k) if k_fastest else (b, k, n))
    old = synth.normal_bf16(80, 2, (b, m, n), 8.0)
    spec = M.Matmul(list(shape), (M.bf16, M.bf16, M.bf16), [None, M.layout(0, 2, 1) if k_fastest else None, None], accum)
    want = run_spec(spec, [A, Bm, old])
    guarded = np.full(old.size + 2, 0x4242, np.uint16)
    guarded[1:-1] = old.ravel()
    bufs = [M.DeviceBuffer.from_numpy(x) for x in (A, Bm, guarded)]
    spec.run_device([bufs[0].ptr, bufs[1].ptr, bufs[2].ptr + 2])
    got = bufs[2].to_numpy(np.uint16, guarded.shape)
    for x in bufs:
        x.free()
    assert np.array_equal(got[1:-1].reshape(old.shape), want) and got[0] == got[-1] == 0x4242
