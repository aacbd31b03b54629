"""First-layer Conv on pixels of three or four channels (conv_pixels.hip) against the oracle."""
import numpy as np
import pytest

import morello_amd as M
import orc
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu
NHWC = orc.make_layout([0, 2, 3, 1])
TYPES = {"u8": ((M.u8, M.i8, M.i32), [0, 1, 5]), "i8": ((M.i8, M.i8, M.i32), [1, 1, 5]), "bf16": ((M.bf16, M.bf16, M.f32), [7, 7, 6])}


@pytest.mark.parametrize("types", ["u8", "i8", "bf16"])
@pytest.mark.parametrize("shape,accum", [
    ((1, 16, 3, 1, 1, 1, 1), False),        # (times 4e5 images below: a single pixel each)
    ((3, 32, 4, 5, 17, 1, 4), True),        # one row of a window, a pixel past an item's edge both ways
    ((2, 48, 3, 4, 16, 2, 3), False),       # whole items, blocks of filters that end inside a group
    ((2, 80, 4, 7, 33, 5, 2), True),        # a second group of one block
    ((1, 96, 3, 30, 31, 3, 8), False),      # eight pixels a row: the widest of bf16
    ((2, 64, 4, 19, 18, 7, 5), True),
    ((1, 16, 3, 21, 15, 6, 6), False),
    ((5, 16, 3, 230, 250, 3, 3), False),    # several items a wave
    ((2, 112, 3, 101, 130, 3, 3), True),    # four groups of 32 filters, the last one half empty
    ((2, 144, 3, 101, 130, 2, 2), False),   # groups of 32, the last of one block
    ((1, 64, 3, 9, 20, 14, 7), False),      # int8: a patch of more pixels than a wave holds in flight
    ((1, 32, 3, 12, 12, 4, 13), True),      # int8: four chunks a row
])
def test_three_and_four_channels(gpu, shape, accum, types):
    """Integers bit for bit, bf16 to 1e-5 of the largest (f32 sums of at most 400 products in another order), from
    operands one element into their buffers; NaN and infinity in a bf16 image reach the outputs whose
    windows hold them and no others."""
    dts, codes = TYPES[types]
    b, f, c, oh, ow, fh, fw = shape
    if (oh, ow) == (1, 1):
        b = 2500
        shape = (b,) + shape[1:]
    gen = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16}
    img, filt = gen[dts[0]](160, 0, (b, oh + fh - 1, ow + fw - 1, c)), gen[dts[1]](160, 1, (f, fh, fw, c))
    out0 = synth.uniform_u8(160, 2, (b, oh, ow, f)).astype(np.float32 if types == "bf16" else np.int32) - 100
    spec = M.Conv(list(shape), dts, accum=accum)
    if types != "bf16" or fw <= 8 and fh * fw <= 49:   # (beyond that, another kernel's)
        assert spec.plan().kernels == ["k_conv_windows"] and spec.plan().steps[0].block[0] == 512

    def run(image, shift):
        held = [np.zeros(x.size + shift, x.dtype) for x in (image, filt)]
        held[0][shift:], held[1][shift:] = image.reshape(-1), filt.reshape(-1)
        bufs = [M.DeviceBuffer.from_numpy(x) for x in held + [out0]]
        spec.run_device([bufs[0].ptr + shift * img.itemsize, bufs[1].ptr + shift * filt.itemsize, bufs[2].ptr])
        got = bufs[2].to_numpy(out0.dtype, out0.shape)
        for x in bufs:
            x.free()
        return got

    want = orc.conv(list(shape), codes, img, filt, out0.copy(), accum, layouts=[NHWC] * 3)
    for shift in (0, 1):
        got = run(img, shift)
        if types != "bf16":
            assert np.array_equal(got, want)
        else:
            assert float(np.abs(got.astype(np.float64) - want).max() / np.abs(want).max()) < 1e-5
    if types == "bf16":
        img = img.copy()
        img[0, 0, 0, 0], img[b - 1, oh + fh - 2, ow + fw - 2, c - 1], img[0, (oh + fh - 1) // 2, (ow + fw - 1) // 2, 1] = 0x7fc0, 0x7f80, 0xff80
        want = orc.conv(list(shape), codes, img, filt, out0.copy(), accum, layouts=[NHWC] * 3)
        got = run(img, 0)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        ok = np.isfinite(want)
        assert not ok.any() or float(np.abs(got[ok].astype(np.float64) - want[ok]).max() / np.abs(want[ok]).max()) < 1e-5


@pytest.mark.parametrize("types", ["u8", "i8", "bf16"])
@pytest.mark.parametrize("fh,fw", [(1, 3), (2, 2), (3, 3), (4, 5), (5, 5), (6, 4), (7, 7), (7, 3), (3, 7)])
@pytest.mark.parametrize("f,c", [(16, 3), (32, 4), (48, 3), (96, 4)])
def test_filters_in_registers(gpu, types, fh, fw, f, c):
    """Every number of filter rows that stays in registers, whole steps and tails, whole cache lines of the output and not; an
    infinity and a NaN in a bf16 image reach the outputs whose windows hold them and no others."""
    dts, codes = TYPES[types]
    b, oh, ow = 2, 21, 37
    shape = [b, f, c, oh, ow, fh, fw]
    gen = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16}
    img, filt = gen[dts[0]](161, 0, (b, oh + fh - 1, ow + fw - 1, c)), gen[dts[1]](161, 1, (f, fh, fw, c))
    if types == "bf16":
        img = img.copy()
        img[0, 0, 0, 0], img[1, oh // 2, ow // 2, 1] = 0x7f80, 0x7fc0
    out0 = synth.uniform_u8(161, 2, (b, oh, ow, f)).astype(np.float32 if types == "bf16" else np.int32) - 100
    for accum in (False, True):
        spec = M.Conv(shape, dts, accum=accum)
        assert spec.plan().kernels == ["k_conv_windows"]
        got = run_spec(spec, [img, filt, out0])
        want = orc.conv(shape, codes, img, filt, out0.copy(), accum, layouts=[NHWC] * 3)
        if types != "bf16":
            assert np.array_equal(got, want)
            continue
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        ok = np.isfinite(want)
        assert float(np.abs(got[ok].astype(np.float64) - want[ok]).max() / np.abs(want[ok]).max()) < 1e-5


def _items(b, oh, ow):
    return b * ((oh + 1) // 2) * ((ow + 15) // 16)


@pytest.mark.parametrize("types", ["u8", "bf16"])
@pytest.mark.parametrize("shape,form", [
    ((60, 64, 3, 41, 53, 7, 7), "held"),     # two and a half items a wave, whole lines
    ((60, 64, 4, 41, 53, 3, 3), "held"),
    ((30, 96, 3, 41, 53, 5, 7), "held"),     # three groups, nearly two items a wave
    ((31, 80, 3, 41, 53, 6, 4), "held"),     # ... the last group half empty: no whole lines
    ((36, 128, 3, 41, 53, 3, 3), "held"),    # below three rounds of waves, all groups counted
    ((55, 128, 3, 41, 53, 3, 3), "shared"),  # past them: one patch for four groups
    ((50, 96, 4, 41, 53, 3, 3), "shared"),   # for three
    ((52, 112, 3, 41, 53, 3, 3), "shared"),  # for four, the last one half empty
])
def test_several_items_a_wave(gpu, types, shape, form):
    """The patch of an item replaces the one before it while the next item's pixels are in flight; filters in registers, or all groups
    of them in LDS against one patch.  Accumulating and not, odd heights and widths."""
    dts, codes = TYPES[types]
    b, f, c, oh, ow, fh, fw = shape
    gen = {M.u8: synth.uniform_u8, M.bf16: synth.normal_bf16}
    img, filt = gen[dts[0]](162, 0, (b, oh + fh - 1, ow + fw - 1, c)), (synth.uniform_i8 if types == "u8" else synth.normal_bf16)(162, 1, (f, fh, fw, c))
    out0 = synth.uniform_u8(162, 2, (b, oh, ow, f)).astype(np.float32 if types == "bf16" else np.int32) - 100
    want = orc.conv(list(shape), codes, img, filt, np.zeros_like(out0), False, layouts=[NHWC] * 3)
    for accum in (False, True):
        spec = M.Conv(list(shape), dts, accum=accum)
        step = spec.plan().steps[0]
        assert spec.plan().kernels == ["k_conv_windows"] and ("RPS = " in step.kernel) == (form == "held"), step
        assert _items(b, oh, ow) > 8 * step.grid[0] and step.grid[1] == (1 if form == "shared" else (f + 31) // 32)
        got = run_spec(spec, [img, filt, out0])
        total = want + out0 if accum else want
        if types == "u8":
            assert np.array_equal(got, total)
        else:   # f32 sums of at most 147 products in another order
            assert float(np.abs(got.astype(np.float64) - total).max() / np.abs(total).max()) < 1e-5


def test_groups_of_64_filters(gpu):
    """bf16 windows of one chunk a row are not held in registers: 144 filters in groups of 64, the last of one block."""
    shape = [4, 144, 3, 101, 130, 2, 2]
    spec = M.Conv(shape, TYPES["bf16"][0])
    step = spec.plan().steps[0]
    assert "RPS = " not in step.kernel and step.grid[1] == 3, step
    img, filt = synth.normal_bf16(163, 0, (4, 102, 131, 3)), synth.normal_bf16(163, 1, (144, 2, 2, 3))
    want = orc.conv(shape, TYPES["bf16"][1], img, filt, np.zeros((4, 101, 130, 144), np.float32), False, layouts=[NHWC] * 3)
    got = run_spec(spec, [img, filt, np.zeros((4, 101, 130, 144), np.float32)])
    assert float(np.abs(got.astype(np.float64) - want).max() / np.abs(want).max()) < 1e-5
