"""Conv as an implicit Matmul on the tiles of gemm_ring_tile.h (conv_gemm.hip), against float64."""
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


@pytest.mark.parametrize("accum", [False, True])
@pytest.mark.parametrize("types,shape,tiles,slices", [
    # [images, filters, channels, height, width of the output, of the filters]
    ("bf16", [3, 5, 48, 8, 5, 3, 3], "RA = 2, RB = 1", 1),        # pixels short of a tile, six steps and three quarters
    ("u8", [1, 34, 32, 7, 4, 5, 5], "RA = 2, RB = 1", 1),         # two filters past a tile
    ("i8", [2, 32, 48, 16, 16, 3, 3], "RA = 2, RB = 1", 1),
    ("bf16", [1, 5, 128, 8, 6, 5, 5], "RA = 2, RB = 1", 6),       # slices of the windows, which end inside their rows
    ("u8", [9, 1, 560, 7, 8, 2, 2], "RA = 2, RB = 1", 2),
    ("bf16", [4, 79, 24, 19, 4, 3, 3], "RA = 2, RB = 2", 1),      # pixels of three chunks
    ("i8", [3, 71, 240, 8, 5, 2, 2], "RA = 2, RB = 2", 1),
    ("u8", [1, 67, 16, 61, 33, 7, 5], "RA = 2, RB = 2", 1),       # pixels of one chunk, filters higher than wide
    ("u8", [1, 76, 160, 5, 19, 5, 5], "RA = 2, RB = 2", 4),
    ("bf16", [10, 4, 264, 50, 33, 2, 2], "RA = 4, RB = 1", 1),
    ("i8", [8, 25, 112, 44, 47, 3, 3], "RA = 4, RB = 1", 1),
    ("bf16", [6, 186, 304, 38, 25, 2, 2], "RA = 4, RB = 2", 1),
    ("u8", [3, 350, 368, 23, 51, 3, 3], "RA = 4, RB = 2", 1),
    ("bf16", [8, 323, 352, 44, 47, 2, 2], "RA = 4, RB = 4", 1),
    ("i8", [6, 133, 352, 49, 53, 3, 3], "RA = 4, RB = 4", 1),
    ("bf16", [4, 263, 368, 57, 59, 2, 2], "RA = 4, RB = 6", 1),
])
def test_windows_on_ring_tiles(gpu, types, shape, tiles, slices, accum):
    """Integers exactly; bf16 within one rounding of 2^-24 of the sum of magnitudes for every term."""
    dts = TYPES[types]
    b, f, c, oh, ow, fh, fw = shape
    spec = M.Conv(shape, dts, accum=accum)
    plan = spec.plan()
    assert f"{tiles}, CONV = true" in plan.steps[0].kernel and plan.steps[0].grid[1] == slices, plan
    assert plan.kernels == ["k_gemm", "k_sum_splits"][:1 + (slices > 1)]
    img, filt = GEN[dts[0]](201, 0, (b, oh + fh - 1, ow + fw - 1, c)), GEN[dts[1]](201, 1, (f, fh, fw, c))
    old = synth.uniform_i8(201, 2, (b, oh, ow, f)).astype(np.int32 if dts[2] == M.i32 else np.float32) * 3
    got = run_spec(spec, [img, filt, old.copy()])
    x, w = _wide(img), _wide(filt)
    want = _conv(x, w, oh, ow) + (old if accum else 0)
    if dts[2] == M.i32:
        assert np.array_equal(got, want.astype(np.int32))
    else:
        k = fh * fw * c
        assert (np.abs(got - want) <= (k + 2) * 2.0 ** -24 * (_conv(np.abs(x), np.abs(w), oh, ow) + 400)).all()


@pytest.mark.parametrize("types,shape", [("i8", [2, 128, 256, 7, 9, 3, 3]), ("bf16", [5, 40, 96, 30, 31, 3, 3])])
def test_windows_on_ring_tiles_and_on_squares_agree(gpu, types, shape):
    """The same Spec through the square tile that an action names."""
    dts = TYPES[types]
    b, f, c, oh, ow, fh, fw = shape
    spec = M.Conv(shape, dts)
    assert "RA = " in spec.plan().steps[0].kernel
    img, filt = GEN[dts[0]](202, 0, (b, oh + fh - 1, ow + fw - 1, c)), GEN[dts[1]](202, 1, (f, fh, fw, c))
    out = np.zeros((b, oh, ow, f), np.int32 if dts[2] == M.i32 else np.float32)
    got = run_spec(spec, [img, filt, out])
    square = [a for a in spec.actions() if a.kind == M.ActionKind.SpatialSplit][0]
    assert "RA = " not in square.plan().steps[0].kernel
    bufs = [M.DeviceBuffer.from_numpy(a) for a in (img, filt, out)]
    square.run_device([x.ptr for x in bufs])
    other = bufs[2].to_numpy(out.dtype, out.shape)
    for x in bufs:
        x.free()
    assert np.array_equal(got, other) if dts[2] == M.i32 else np.allclose(got, other, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("types,shape,tiles", [
    ("u8", [7, 272, 16, 72, 72, 3, 3], "RA = 4, RB = 2"),     # two steps, the second an eighth full; 256 x 256 tiles otherwise
    ("i8", [9, 258, 48, 61, 67, 1, 3], "RA = 4, RB = 2"),     # filters lower than wide, two past a tile
    ("u8", [1, 48, 64, 21, 21, 5, 5], "RA = 2, RB = 1"),
    ("bf16", [21, 61, 144, 17, 17, 3, 3], "RA = 2, RB = 2"),  # the last row of tiles 53 pixels, its last column 61 filters
])
def test_windows_straight_into_lds(gpu, types, shape, tiles):
    test_windows_on_ring_tiles(gpu, types, shape, tiles, 1, True)
