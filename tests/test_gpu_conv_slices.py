"""Conv as an implicit Matmul whose windows are shared out in slices that are not all equal."""
import numpy as np
import pytest

import morello_amd as M
import orc
from gpu_util import run_spec
from morello_amd import synth

pytestmark = pytest.mark.gpu

NHWC = orc.make_layout([0, 2, 3, 1])
TYPES = {"u8": ((M.u8, M.i8, M.i32), [0, 1, 5], 1), "i8": ((M.i8, M.i8, M.i32), [1, 1, 5], 1),
         "bf16": ((M.bf16, M.bf16, M.f32), [7, 7, 6], 2), "f32": ((M.f32, M.f32, M.f32), [6, 6, 6], 4)}
GEN = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16, M.f32: synth.normal_f32}


@pytest.mark.parametrize("types", list(TYPES))
@pytest.mark.parametrize("channel_bytes,fh,fw", [
    (544, 5, 5),   # 106 steps of 128 bytes and a quarter
    (688, 3, 3),   # 48 and 48 bytes
    (256, 3, 3),   # 18 whole ones: halves
    (352, 3, 3),   # 25, in slices of nine, nine and seven
    (80, 5, 5),    # 15 and 80 bytes: the last slice ends in a part of a step
    (16, 11, 11),  # 15 and 16 bytes, pixels of a single chunk
])
@pytest.mark.parametrize("accum", [False, True])
def test_slices_of_unequal_length(gpu, types, channel_bytes, fh, fw, accum):
    """The last slice shorter than the others or ending inside a step; integers exactly, floats to
    the rounding of sums of this length, an infinity in the last channel of the last window kept."""
    dts, codes, size = TYPES[types]
    b, f, c, oh, ow = 2, 40, channel_bytes // size, 5, 7
    shape = [b, f, c, oh, ow, fh, fw]
    spec = M.Conv(shape, dts, accum=accum)
    plan = spec.plan()
    assert plan.kernels == ["k_gemm", "k_sum_splits"] and plan.steps[0].grid[1] > 1
    img, filt = GEN[dts[0]](171, 0, (b, oh + fh - 1, ow + fw - 1, c)), GEN[dts[1]](171, 1, (f, fh, fw, c))
    if types == "bf16":
        img = img.copy()
        img[1, oh + fh - 2, ow + fw - 2, c - 1] = 0x7f80
    out_np = np.float32 if size > 1 else np.int32
    out0 = synth.uniform_u8(171, 2, (b, oh, ow, f)).astype(out_np) - 100
    got = run_spec(spec, [img, filt, out0.copy()])
    want = orc.conv(shape, codes, img, filt, out0.copy(), accum, layouts=[NHWC] * 3)
    if size == 1:
        assert np.array_equal(got, want)
        return
    assert np.array_equal(np.isinf(got), np.isinf(want)) and not np.isnan(got).any()
    ok = np.isfinite(want)
    assert float(np.abs(got[ok].astype(np.float64) - want[ok]).max() / np.abs(want[ok]).max()) < 1e-5
