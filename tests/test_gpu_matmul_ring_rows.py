"""Matmuls of rows that start anywhere, read in place (gemm_ring_rows.hip), against float64."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu
KT = M.layout(0, 2, 1)
TYPES = {"u8": (M.u8, M.i8, M.i32), "i8": (M.i8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.f32), "bf16_out": (M.bf16, M.bf16, M.bf16)}
GEN = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16}


def _widen(x):
    return (x.astype(np.uint32) << 16).view(np.float32) if x.dtype == np.uint16 else x


def _check(got, A, B, C, accum, dts):
    """Integers exactly; bf16 within k rounding errors of 2^-24 of the sum of magnitudes, a bf16 result rounded once."""
    a64, b64 = _widen(A).astype(np.float64), _widen(B).astype(np.float64)
    want = a64 @ b64 + (_widen(C).astype(np.float64) if accum else 0)
    if dts[2] == M.i32:
        assert np.array_equal(got, want.astype(np.int32))
        return
    diff = np.abs(_widen(got).astype(np.float64) - want)
    bound = (A.shape[2] + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + 8)
    assert (diff <= bound + (2.0 ** -8 * np.abs(want) if dts[2] == M.bf16 else 0)).all()


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("types", list(TYPES))
@pytest.mark.parametrize("b,m,k_bytes,n,accum,families", [
    (1, 1900, 3 * 128 + 2, 487, False, 1),   # one element in the first step
    (1, 900, 4 * 128 - 2, 1025, True, 1),    # one short of four whole steps
    (3, 65, 9 * 128 + 6, 707, False, 1),     # a row past a tile, three columns of the last one its own
    (2, 384, 5 * 128 + 62, 577, True, 1),    # whole tiles in m; one column
    (1, 191, 40 * 128 + 34, 133, False, 2),  # slices of K, the last one shorter
    (1, 100, 33 * 128 + 18, 250, True, 2),   # ... the old values added in the sum
    (2, 641, 6 * 128 + 14, 1027, True, 1),   # tiles of 128 x 64
    (1, 1283, 8 * 128 + 30, 1021, False, 1),
    (1, 461, 15 * 128, 656, True, 1),        # rows of whole chunks
    (2, 200, 9 * 128 + 16, 336, False, 1),
    (1, 1000, 1000, 1000, False, 1),         # one round of tiles to the last
    (1, 384, 2558, 120, False, 1),           # fewer than 128 columns
    (2, 1270, 130, 210, True, 1),            # two steps
    (1, 1300, 270, 690, False, 1),           # three
])
def test_rows_that_start_anywhere(gpu, b, m, k_bytes, n, accum, families, types, nk):
    dts = TYPES[types]
    k = k_bytes // (2 if dts[0] == M.bf16 else 1)
    A, B = GEN[dts[0]](181, 0, (b, m, k)), GEN[dts[1]](181, 1, (b, k, n))
    C = {M.i32: lambda: synth.uniform_i8(181, 2, (b, m, n)).astype(np.int32) * 1001,
         M.f32: lambda: synth.normal_f32(181, 2, (b, m, n)), M.bf16: lambda: synth.normal_bf16(181, 2, (b, m, n))}[dts[2]]()
    spec = M.Matmul([b, m, k, n], dts, [None, KT if nk else None, None], accum)
    plan = spec.plan()
    assert plan.kernels == ["k_gemm_ring", "k_sum_splits"][:families], plan
    assert plan.steps[0].grid[1] > b or families == 1
    stored = np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B
    _check(run_spec(spec, [A, stored, C.copy()]), A, B, C, accum, dts)
    # the same at addresses an element past an aligned one
    held = [np.zeros(x.size + 1, x.dtype) for x in (A, stored, C)]
    for h, x in zip(held, (A, stored, C)):
        h[1:] = x.reshape(-1)
    bufs = [M.DeviceBuffer.from_numpy(h) for h in held]
    spec.run_device([d.ptr + h.itemsize for d, h in zip(bufs, held)])
    got = bufs[2].to_numpy(C.dtype, held[2].shape)
    assert got[0] == 0
    _check(got[1:].reshape(C.shape), A, B, C, accum, dts)
    for d in bufs:
        d.free()


@pytest.mark.parametrize("types", list(TYPES))
@pytest.mark.parametrize("m,k_bytes,n,accum,families", [
    (33, 61 * 128 + 22, 1475, True, 2),      # half a tile of rows, K in slices
    (64, 9 * 128 + 16, 9999, False, 1),      # a whole one, in one piece; rows of whole chunks
])
def test_33_to_64_rows_against_a_large_b(gpu, types, m, k_bytes, n, accum, families):
    dts = TYPES[types]
    k = k_bytes // (2 if dts[0] == M.bf16 else 1)
    A, B = GEN[dts[0]](184, 0, (1, m, k)), GEN[dts[1]](184, 1, (1, k, n))
    C = {M.i32: lambda: synth.uniform_i8(184, 2, (1, m, n)).astype(np.int32) * 1001,
         M.f32: lambda: synth.normal_f32(184, 2, (1, m, n)), M.bf16: lambda: synth.normal_bf16(184, 2, (1, m, n))}[dts[2]]()
    spec = M.Matmul([1, m, k, n], dts, [None, KT, None], accum)
    assert spec.plan().kernels == ["k_gemm_ring", "k_sum_splits"][:families]
    _check(run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)), C.copy()]), A, B, C, accum, dts)


@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("types,m,k,n", [("bf16", 1411, 733, 1555), ("bf16_out", 1300, 1501, 2049), ("bf16_out", 1153, 201, 1861), ("bf16", 1153, 65, 1861)])
def test_tiles_of_128_columns(gpu, types, m, k, n, nk):
    dts = TYPES[types]
    A, B = synth.normal_bf16(182, 0, (1, m, k)), synth.normal_bf16(182, 1, (1, k, n))
    C = np.zeros((1, m, n), np.uint16 if dts[2] == M.bf16 else np.float32)
    spec = M.Matmul([1, m, k, n], dts, [None, KT if nk else None, None])
    assert spec.plan().kernels == ["k_gemm_ring"]
    _check(run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, C]), A, B, C, False, dts)


@pytest.mark.parametrize("types,b,m,k,n,columns,orders,accum", [
    ("bf16", 1, 1411, 733, 2733, 160, "kn nk", False),       # rows and columns short of a tile, odd rows of both
    ("bf16_out", 2, 641, 898, 3203, 160, "kn nk", True),     # a row and three columns past one; rows on words
    ("bf16", 1, 2432, 386, 1840, 160, "kn nk", True),        # whole tiles but the last column's half; two elements past six steps
    ("bf16_out", 1, 1500, 449, 3649, 192, "kn nk", False),   # one column past a tile, one element past seven steps
    ("bf16", 1, 2305, 1024, 2307, 192, "kn", True),          # rows of A of whole chunks
    ("bf16_out", 1, 1185, 2047, 3370, 160, "kn", False),     # the longest K, odd rows
    ("bf16", 1, 1281, 2942, 1997, 128, "kn", False),     # ... on the smaller tile, rows on words
])
def test_tiles_past_a_round_of_128_columns(gpu, types, b, m, k, n, columns, orders, accum):
    dts = TYPES[types]
    A, B = synth.normal_bf16(185, 0, (b, m, k)), synth.normal_bf16(185, 1, (b, k, n))
    C = synth.normal_bf16(185, 2, (b, m, n)) if dts[2] == M.bf16 else synth.normal_f32(185, 2, (b, m, n))
    for order in orders.split():
        nk = order == "nk"
        spec = M.Matmul([b, m, k, n], dts, [None, KT if nk else None, None], accum)
        plan = spec.plan()
        assert plan.kernels == ["k_gemm_ring"] and plan.steps[0].grid[0] == -(-m // 128) * -(-n // columns), plan
        _check(run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, C.copy()]), A, B, C, accum, dts)


@pytest.mark.parametrize("types,b,m,k,n,columns,nk,accum", [
    ("u8", 1, 1285, 522, 1537, 128, True, False),    # ten bytes past four steps, rows on pairs of bytes
    ("i8", 1, 1281, 4348, 1537, 128, True, True),    # the longest K, rows on words
    ("u8", 2, 641, 770, 3203, 160, True, True),
    ("u8", 1, 2432, 642, 1840, 160, False, True),    # whole tiles but the last column's half
    ("i8", 1, 1500, 1030, 3649, 192, False, False),  # one column past a tile
    ("u8", 1, 1500, 1030, 3649, 192, True, False),
])
def test_int8_tiles_past_a_round(gpu, types, b, m, k, n, columns, nk, accum):
    dts = TYPES[types]
    A, B = GEN[dts[0]](186, 0, (b, m, k)), GEN[dts[1]](186, 1, (b, k, n))
    C = synth.uniform_i8(186, 2, (b, m, n)).astype(np.int32) * 1001
    spec = M.Matmul([b, m, k, n], dts, [None, KT if nk else None, None], accum)
    plan = spec.plan()
    assert plan.kernels == ["k_gemm_ring"] and plan.steps[0].grid[0] == -(-m // 128) * -(-n // columns), plan
    _check(run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, C.copy()]), A, B, C, accum, dts)


def test_nonfinite_operands_stay_in_their_rows_and_columns(gpu):
    """A NaN and infinities beside the ends of K, M and N, and of the first step, reach the rows and columns that hold them only."""
    for m, k, n in ((129, 733, 1195), (129, 3333, 195)):   # whole, and in slices of K
        A, B = synth.normal_bf16(183, 0, (1, m, k)), synth.normal_bf16(183, 1, (1, k, n))
        A[0, 7, k - 1], A[0, m - 1, 0], B[0, k - 1, n - 1], B[0, k % 64, 3], A[0, 64, k % 64] = 0x7fc0, 0x7f80, 0xff80, 0x7f80, 0x7fc0
        for nk in (False, True):
            spec = M.Matmul([1, m, k, n], TYPES["bf16"], [None, KT if nk else None, None])
            assert spec.plan().kernels[0] == "k_gemm_ring"
            got = run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, np.zeros((1, m, n), np.float32)])
            finite = np.ones((m, n), bool)
            finite[7], finite[64], finite[m - 1], finite[:, n - 1], finite[:, 3] = False, False, False, False, False
            assert np.array_equal(np.isfinite(got[0]), finite)
