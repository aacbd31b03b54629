"""Moves whose two sides share their contiguous digit, in whole vectors (k_move_runs), and the edges of
the gather kernel's runs of four, bit for bit against the CPU oracle."""
import numpy as np
import pytest

import morello_amd as M
import orc
from morello_amd import synth

pytestmark = pytest.mark.gpu

NP = {M.u8: np.uint8, M.i8: np.int8, M.u16: np.uint16, M.i32: np.int32, M.f32: np.float32, M.bf16: np.uint16}


def _values(dt, shape):
    if dt == M.f32:
        x = (synth.normal_f32(850, 0, shape) * 300).astype(np.float32)
        x.reshape(-1)[:4] = [np.nan, np.inf, -0.0, 1e20]
        return x
    if dt == M.bf16:
        return synth.normal_bf16(850, 1, shape, 100.0)
    return synth.raw_u64(850, 2, int(np.prod(shape))).astype(NP[dt]).reshape(shape)


def _layouts(dims):
    if dims is None:
        return None, None
    m = [(d[0], (M.Packed if d[1] == "p" else M.OddEven)(d[2])) if isinstance(d, tuple) else d for d in dims]
    o = [(d[0], 1 if d[1] == "p" else 2, d[2]) if isinstance(d, tuple) else d for d in dims]
    return M.layout(*m), orc.make_layout(o)


def _check(sdt, ddt, shape, src, dst, kernel, shift=(0, 0)):
    """`shift`: elements by which the two buffers start past an aligned address."""
    (ls, lso), (ld, ldo) = _layouts(src), _layouts(dst)
    spec = M.Move(shape, (sdt, ddt), layouts=[ls, ld])
    assert spec.plan().kernels == [kernel]   # (for aligned buffers: a plan knows no addresses)
    x, n = _values(sdt, shape), int(np.prod(shape))
    guard = np.full(n + 2 * shift[1] + 16, 0x5a, NP[ddt])   # what lies around the result stays
    held = np.zeros(n + shift[0], NP[sdt])
    held[shift[0]:] = x.reshape(-1)
    a, b = M.DeviceBuffer.from_numpy(held), M.DeviceBuffer.from_numpy(guard)
    spec.run_device([a.ptr + shift[0] * x.itemsize, b.ptr + shift[1] * guard.itemsize])
    got = b.to_numpy(guard.dtype, guard.shape)
    want = orc.move(shape, [int(sdt), int(ddt)], x, np.zeros(n, NP[ddt]), layouts=[lso, ldo])
    assert np.array_equal(got[shift[1]:shift[1] + n].view(np.uint8), want.reshape(-1).view(np.uint8))
    assert (got[:shift[1]] == 0x5a).all() and (got[shift[1] + n:] == 0x5a).all()
    a.free()
    b.free()


STRIPS = (0, 2, 1, (2, "p", 16))


@pytest.mark.parametrize("sdt,ddt", [(M.f32, M.bf16), (M.f32, M.f32), (M.bf16, M.f32), (M.u8, M.f32), (M.u8, M.bf16),
                                     (M.bf16, M.u8), (M.i32, M.u8)])
@pytest.mark.parametrize("rows,cols", [(2, 32), (3, 16 * 7), (129, 16 * 33), (700, 16 * 80), (37, 16 * 600)])
def test_packing_strips(gpu, sdt, ddt, rows, cols):
    """Strips of 16 columns, converted and not, from a single vector's neighbourhood over ragged tiles (257 vectors a
    side) up to tiles of four vectors a thread, and back."""
    _check(sdt, ddt, [1, rows, cols], None, STRIPS, "k_move_runs")
    _check(ddt, sdt, [1, rows, cols], STRIPS, None, "k_move_runs")


@pytest.mark.parametrize("dt,pack", [(M.bf16, 4), (M.bf16, 2), (M.u8, 8), (M.u8, 4), (M.f32, 2), (M.i32, 4)])
def test_runs_shorter_than_a_vector(gpu, dt, pack):
    """Packed digits of 4, 8 and 16 bytes: the narrower vectors."""
    _check(dt, dt, [1, 67, 24 * pack], None, (0, 2, 1, (2, "p", pack)), "k_move_runs" if pack * np.dtype(NP[dt]).itemsize >= 8 else "k_move_rows")


@pytest.mark.parametrize("shift", [(1, 0), (0, 1), (2, 2), (4, 4), (8, 4)])
def test_buffers_off_a_vector(gpu, shift):
    """Buffers that start on any element: the widest vector both sides allow, else the kernel without vectors."""
    _check(M.f32, M.bf16, [1, 150, 320], None, STRIPS, "k_move_runs", shift)


def test_long_shared_digit_is_cut(gpu):
    """A shared digit longer than 256 vectors, in pieces of even length; five digits."""
    _check(M.f32, M.f32, [6, 5, 1028 * 4], None, (1, 0, 2), "k_move_runs")
    _check(M.u8, M.f32, [3, 4, 5, 6, 64], None, (3, 0, 2, 1, 4), "k_move_runs")


@pytest.mark.parametrize("sdt,ddt", [(M.u8, M.f32), (M.bf16, M.f32), (M.u8, M.u8), (M.f32, M.bf16)])
@pytest.mark.parametrize("rows,cols,dst", [(1024, 272, (0, 1, 2, (2, "oe", 16))), (1040, 99, (0, 1, 2, (1, "p", 16))),
                                           (1168, 130, (0, 1, 2, (1, "p", 16))), (4096, 48, (0, 2, 1, (1, "oe", 4)))])
def test_gathered_runs_of_four(gpu, sdt, ddt, rows, cols, dst):
    """Even and odd elements apart, strips of rows over odd widths: runs of four on one side, both or none."""
    _check(sdt, ddt, [1, rows, cols], None, dst, "k_move_gather")


@pytest.mark.parametrize("sdt,ddt", [(M.f32, M.bf16), (M.f32, M.f32), (M.bf16, M.f32), (M.u8, M.f32), (M.u8, M.bf16),
                                     (M.bf16, M.u8), (M.i32, M.u8)])
@pytest.mark.parametrize("rows,cols", [(1030, 16 * 65), (1027, 16 * 129), (2049, 16 * 130)])
def test_packing_strips_in_tiles(gpu, sdt, ddt, rows, cols):
    """Past the 2^20 elements up to which a vector goes to a thread: tiles of one and of four vectors a thread,
    ragged on both sides."""
    _check(sdt, ddt, [1, rows, cols], None, STRIPS, "k_move_runs")
    _check(ddt, sdt, [1, rows, cols], STRIPS, None, "k_move_runs")


def test_long_runs_without_tiles(gpu):
    """Whole vectors in runs of 64 bytes and more, up to 16 MB; and beyond, in tiles."""
    _check(M.f32, M.f32, [7340, 12, 16], None, (1, 0, 2), "k_move_runs")
    _check(M.u8, M.u8, [30, 14, 5, 8, 260], (0, 2, 1, 3, 4), (1, 2, 0, 3, 4), "k_move_runs")
    _check(M.f32, M.f32, [29360, 12, 16], None, (1, 0, 2), "k_move_runs")


@pytest.mark.parametrize("shift", [(1, 0), (0, 1), (2, 2), (4, 4), (8, 4)])
def test_tiles_off_a_vector(gpu, shift):
    _check(M.f32, M.bf16, [1, 1050, 1040], None, STRIPS, "k_move_runs", shift)


@pytest.mark.parametrize("sdt,ddt", [(M.f32, M.f32), (M.f32, M.bf16), (M.bf16, M.bf16), (M.u8, M.f32)])
def test_five_digits_short_and_long(gpu, sdt, ddt):
    """More digits than a tile has: four of them short (no tile), and two on the source side before its runs are
    long."""
    _check(sdt, ddt, [20011, 2, 2, 2, 8], None, (0, 3, 2, 1, 4), "k_move_runs")
    _check(sdt, ddt, [20011, 3, 2, 2, 16], None, (3, 0, 2, 1, 4), "k_move_runs")
    _check(sdt, ddt, [107, 4, 696, 4, 4], None, (4, 3, 2, 1, 0, (4, "p", 2)), "k_move_runs" if max(np.dtype(NP[sdt]).itemsize, np.dtype(NP[ddt]).itemsize) == 4 else "k_move_gather")
    _check(sdt, ddt, [2, 58566, 4, 3, 8], (0, 3, 1, 2, 4), (1, 0, 2, 3, 4), "k_move_runs")


@pytest.mark.parametrize("sdt,ddt", [(M.u8, M.f32), (M.bf16, M.f32), (M.u8, M.u8), (M.f32, M.bf16), (M.bf16, M.bf16), (M.f32, M.f32)])
@pytest.mark.parametrize("shape,src,dst", [
    ([18, 60002], None, (1, 0)), ([18, 60004], None, (1, 0)), ([20, 60002], None, (1, 0)), ([17, 62003], None, (1, 0)),   # 2 and 2, 4 and 2, 2 and 4, none
    ([1189, 5, 2, 4, 26], None, (3, 4, 0, 2, 1, (3, "oe", 2))),   # five digits
    ([6, 7001, 5, 6], (2, 1, 3, 0), (0, 2, 3, 1)), ([3, 6, 30002, 2], (2, 3, 0, 1), (0, 1, 3, 2)),
])
def test_gathered_runs_of_four_and_of_two(gpu, sdt, ddt, shape, src, dst):
    """Past the 2^20 elements up to which an element goes to a thread: every pair of run lengths."""
    _check(sdt, ddt, shape, src, dst, "k_move_gather")


@pytest.mark.parametrize("shift", [(1, 0), (0, 1), (2, 2), (2, 1)])
def test_gathered_runs_off_an_element(gpu, shift):
    _check(M.f32, M.f32, [20, 60004], None, (1, 0), "k_move_gather", shift)
    _check(M.bf16, M.bf16, [20, 60004], None, (1, 0), "k_move_gather", shift)


@pytest.mark.parametrize("sdt,ddt", [(M.f32, M.bf16), (M.i32, M.u16), (M.f32, M.u16)])
@pytest.mark.parametrize("rows,cols,strips,shift", [(1030, 2048, 16, (0, 0)), (513, 2048, 8, (0, 0)), (1030, 1024, 16, (0, 0)), (2049, 3072, 16, (0, 0)), (1025, 2048, 24, (0, 0)),
                                                    (1030, 2048, 16, (4, 0)), (1030, 2048, 16, (0, 4)), (1030, 2048, 16, (2, 8))])
def test_narrowing_rows_8_kib_apart(gpu, sdt, ddt, rows, cols, strips, shift):
    """Rows of multiples of 8 KiB (and of 4 and 12), 32-bit elements to 16-bit ones: eight elements a vector where both buffers are aligned for it, four or two otherwise."""
    if strips == 24:   # a digit between the strips and the rows
        _check(sdt, ddt, [5, rows // 5, cols], None, (2, 1, 0, (2, "p", 8)), "k_move_runs", shift)
    else:
        _check(sdt, ddt, [1, rows, cols], None, (0, 2, 1, (2, "p", strips)), "k_move_runs", shift)


@pytest.mark.parametrize("sdt,ddt", [(M.f32, M.bf16), (M.f32, M.f32), (M.bf16, M.bf16)])
@pytest.mark.parametrize("rows,cols", [(2051, 16 * 512), (4100, 16 * 256)])
def test_packing_strips_along_diagonals(gpu, sdt, ddt, rows, cols):
    """From 64 MB on, both sides together, with rows whole pages apart, tiles are numbered along the source's rows, each row one tile further on: whole and ragged
    rows, more rows of tiles than columns and fewer."""
    _check(sdt, ddt, [1, rows, cols], None, STRIPS, "k_move_runs")
    _check(sdt, ddt, [rows, 128, cols // 128], None, (1, 0, 2), "k_move_runs")
