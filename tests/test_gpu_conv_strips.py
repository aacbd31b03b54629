"""First-layer Conv over strips of several output rows (conv_pixels.hip), against float64: strips of every height that the choice takes, ragged ends of
images and rows, images and filters that start on any element, accumulation."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu
TYPES = {"u8": (M.u8, M.i8, M.i32), "i8": (M.i8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.f32)}
GEN = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16}


def _wide(x):
    return ((x.astype(np.uint32) << 16).view(np.float32) if x.dtype == np.uint16 else x).astype(np.float64)


def _conv(img, filt, oh, ow):
    b, c, (f, fh, fw) = img.shape[0], img.shape[3], filt.shape[:3]
    out = np.zeros((b * oh * ow, f))
    for r in range(fh):
        for s in range(fw):
            out += np.ascontiguousarray(img[:, r:r + oh, s:s + ow]).reshape(-1, c) @ filt[:, r, s].T
    return out.reshape(b, oh, ow, f)


@pytest.mark.parametrize("types,shape", [
    # [images, filters, channels, height, width of the output, of the filters]
    ("bf16", [26, 16, 3, 32, 146, 1, 3]), ("bf16", [15, 16, 3, 141, 56, 3, 3]), ("bf16", [9, 16, 4, 157, 81, 2, 7]), ("bf16", [18, 16, 3, 155, 36, 6, 4]),
    ("bf16", [14, 16, 3, 60, 69, 5, 5]), ("bf16", [9, 16, 4, 165, 33, 7, 7]), ("bf16", [16, 64, 3, 109, 109, 7, 7]), ("bf16", [10, 80, 3, 115, 115, 7, 7]),
    ("u8", [16, 16, 3, 138, 49, 1, 3]), ("u8", [12, 16, 4, 115, 86, 3, 5]), ("u8", [10, 16, 3, 169, 69, 5, 5]), ("u8", [26, 16, 4, 84, 52, 7, 7]),
    ("u8", [3, 96, 3, 174, 174, 5, 5]), ("i8", [28, 16, 3, 105, 39, 1, 3]), ("i8", [26, 16, 4, 108, 34, 5, 5]), ("i8", [23, 16, 3, 89, 52, 7, 7]),
])
@pytest.mark.parametrize("accum", [False, True])
def test_strips(gpu, types, shape, accum):
    """Integers exactly; bf16 within one rounding of 2^-24 of the sum of magnitudes for every term.  The strips' height follows from the shape, three rows to twelve."""
    dts = TYPES[types]
    b, f, c, oh, ow, fh, fw = shape
    spec = M.Conv(shape, dts, accum=accum)
    assert "STRIPS = true" in spec.plan().steps[0].kernel, spec.plan()
    img, filt = GEN[dts[0]](931, 0, (b, oh + fh - 1, ow + fw - 1, c)), GEN[dts[1]](931, 1, (f, fh, fw, c))
    old = synth.uniform_i8(931, 2, (b, oh, ow, f)).astype(np.int32 if dts[2] == M.i32 else np.float32) * 3
    got = run_spec(spec, [img, filt, old.copy()])
    x, w = _wide(img), _wide(filt)
    want = _conv(x, w, oh, ow) + (old if accum else 0)
    if dts[2] == M.i32:
        assert np.array_equal(got, want.astype(np.int32))
    else:
        assert (np.abs(got - want) <= (fh * fw * c + 2) * 2.0 ** -24 * (_conv(np.abs(x), np.abs(w), oh, ow) + 400)).all()


@pytest.mark.parametrize("types,shape", [("bf16", [9, 16, 3, 165, 35, 7, 7]), ("u8", [10, 16, 3, 169, 69, 5, 5])])
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_strips_of_images_off_a_word(gpu, types, shape, shift):
    dts = TYPES[types]
    b, f, c, oh, ow, fh, fw = shape
    spec = M.Conv(shape, dts)
    img, filt = GEN[dts[0]](932, 0, (b, oh + fh - 1, ow + fw - 1, c)), GEN[dts[1]](932, 1, (f, fh, fw, c))
    want = run_spec(spec, [img, filt, np.zeros((b, oh, ow, f), np.int32 if dts[2] == M.i32 else np.float32)])
    bufs = [M.DeviceBuffer.from_numpy(np.concatenate([np.zeros(shift, a.dtype), a.reshape(-1)])) for a in (img, filt)] + [M.DeviceBuffer.from_numpy(np.zeros_like(want))]
    spec.run_device([bufs[0].ptr + shift * img.itemsize, bufs[1].ptr + shift * filt.itemsize, bufs[2].ptr])
    assert np.array_equal(bufs[2].to_numpy(want.dtype, want.shape), want)
    for v in bufs:
        v.free()
