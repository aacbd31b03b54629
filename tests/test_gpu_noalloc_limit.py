"""mrl_run_noalloc near the end of its fixed scratch: copies that do not fit with their rows padded to cache
lines, their K to whole chunks, or a right operand's short columns in chunks, are made smaller."""
import numpy as np
import pytest

import morello_amd as M
from gpu_util import run_spec
from morello_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dts,shape,k_fastest", [
    ((M.u8, M.i8, M.i32), [1, 56000, 515, 16], False),            # rows of 528 bytes fit, of 640 do not
    ((M.bf16, M.bf16, M.f32), [1, 5900, 2817, 640], False),       # 5648, 5760
    ((M.u8, M.i8, M.i32), [2, 40, 3, 1200000], True),             # 2.4 million columns of three bytes, as six rows
])
def test_copies_fit_that_did(gpu, dts, shape, k_fastest):
    b, m, k, n = shape
    spec = M.Matmul(shape, dts, layouts=[None, M.layout(0, 2, 1) if k_fastest else None, None])
    assert spec.plan().scratch_bytes > M.NOALLOC_SCRATCH_BYTES
    bt = (b, n, k) if k_fastest else (b, k, n)
    if dts[0] == M.u8:
        arrays = [synth.uniform_u8(950, 0, (b, m, k)), synth.uniform_i8(950, 1, bt), np.zeros((b, m, n), np.int32)]
    else:
        arrays = [synth.normal_bf16(950, 0, (b, m, k)), synth.normal_bf16(950, 1, bt), np.zeros((b, m, n), np.float32)]
    want = run_spec(spec, arrays)
    bufs = [M.DeviceBuffer.from_numpy(a) for a in arrays]
    spec.run_noalloc([x.ptr for x in bufs])
    M.synchronize()
    got = bufs[2].to_numpy(arrays[2].dtype, arrays[2].shape)
    for x in bufs:
        x.free()
    if dts[2] == M.i32:
        assert np.array_equal(got, want)
    else:
        # the same kernel family over a K that ends elsewhere: f32 sums of 2817 products in another order
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()


def test_conv_fits_without_partial_results(gpu):
    """Windows shared out in slices of unequal length, 10 MB of partial results beside 30 MB of copies to channels-last."""
    b, f, c, oh, fh = 4, 256, 3056, 36, 3
    row_major = M.layout(0, 1, 2, 3)
    spec = M.Conv([b, f, c, oh, oh, fh, fh], [M.u8, M.i8, M.i32], [row_major] * 3)
    assert spec.plan().scratch_bytes > M.NOALLOC_SCRATCH_BYTES
    ih = oh + fh - 1
    arrays = [synth.uniform_u8(951, 0, (b, c, ih, ih)), synth.uniform_i8(951, 1, (f, c, fh, fh)), np.zeros((b, f, oh, oh), np.int32)]
    want = run_spec(spec, arrays)
    bufs = [M.DeviceBuffer.from_numpy(a) for a in arrays]
    spec.run_noalloc([x.ptr for x in bufs])
    M.synchronize()
    got = bufs[2].to_numpy(np.int32, arrays[2].shape)
    for x in bufs:
        x.free()
    assert np.array_equal(got, want)


def test_attention_of_few_queries_fits_without_partial_results(gpu):
    """Padded copies of K and V (33 MB) leave no room for shares of the keys: the same form with one share, which needs none."""
    b, m, keys, d = 8, 16, 8100, 100
    spec = M.ComposeMSM(b, m, d, keys, d, layouts=[None, None, M.layout(0, 2, 1), None])
    one_share = M.Action(spec, M._binding.ActionC(M.ActionKind.Fused, 0, 0, 0, 1, 0, 0, 0, 0.0))
    assert "W = 8" in one_share.plan().steps[-1].kernel
    assert spec.plan().scratch_bytes > M.NOALLOC_SCRATCH_BYTES >= one_share.plan().scratch_bytes
    arrays = [synth.normal_bf16(952, i, s, 0.4) for i, s in enumerate([(b, keys, d), (b, m, d), (b, keys, d)])] + [np.zeros((b, m, d), np.float32)]
    want = run_spec(one_share, arrays)
    bufs = [M.DeviceBuffer.from_numpy(a) for a in arrays]
    spec.run_noalloc([x.ptr for x in bufs])
    M.synchronize()
    got = bufs[3].to_numpy(np.float32, arrays[3].shape)
    for x in bufs:
        x.free()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("shape", [(2, 100, 2761, 8190), (1, 200, 2761, 8190)])
def test_odd_rows_fit_without_copies(gpu, shape):
    """Rows of an odd number of bf16 that go through copies of 47 and 93 MB where there is room are read in place where there is none."""
    b, m, k, n = shape
    spec = M.Matmul(list(shape), (M.bf16, M.bf16, M.f32), layouts=[None, M.layout(0, 2, 1), None])
    assert spec.plan().scratch_bytes > M.NOALLOC_SCRATCH_BYTES
    arrays = [synth.normal_bf16(953, 0, (b, m, k)), synth.normal_bf16(953, 1, (b, n, k)), np.zeros((b, m, n), np.float32)]
    want = run_spec(spec, arrays)
    bufs = [M.DeviceBuffer.from_numpy(a) for a in arrays]
    spec.run_noalloc([x.ptr for x in bufs])
    M.synchronize()
    got = bufs[2].to_numpy(np.float32, arrays[2].shape)
    for x in bufs:
        x.free()
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()   # f32 sums of 2761 products in another order
