"""Which products take k_gemm_ring, and with which tile (gemm_ring.hip): sizes on both sides of each line, against float64."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu


def _widen(x):
    return (x.astype(np.uint32) << 16).view(np.float32) if x.dtype == np.uint16 else x


@pytest.mark.parametrize("types,b,m,k,n,columns", [
    ("bf16", 1, 1153, 832, 896, 64),       # 13 steps of 64, 266 tiles of 64 x 64
    ("bf16", 1, 1153, 768, 896, 0),        # twelve
    ("bf16", 2, 1153, 776, 449, 64),       # the thirteenth an eighth full, odd rows of C
    ("u8", 1, 1153, 1792, 896, 64),        # 14 steps of 128
    ("u8", 1, 1153, 1664, 896, 0),
    ("u8", 2, 1153, 1680, 449, 64),
    ("bf16", 1, 1985, 1792, 1153, 128),    # 28 steps, 160 tiles of 128 x 128, the last row and column of them one wide
    ("bf16", 1, 1985, 1728, 1153, 0),
    ("u8", 1, 1985, 3584, 1153, 128),
    ("u8", 1, 1985, 3456, 1153, 0),
    ("u8", 1, 1984, 3457, 1152, 128),      # of copied rows
    ("i8", 1, 2048, 3472, 2048, 128),      # a whole round
    ("bf16", 1, 704, 2304, 2944, 128),     # 36 steps; 506 tiles of 64 x 64, 276 of 128 x 64, 138 of 128 x 128
    ("bf16", 1, 704, 2240, 2944, 0),
    ("u8", 3, 300, 4593, 1793, 128),
])
@pytest.mark.parametrize("nk", [False, True])
@pytest.mark.parametrize("accum", [False, True])
def test_widths(gpu, types, b, m, k, n, columns, nk, accum):
    """Integers exact; bf16 sums of k products in f32 are within k rounding errors of 2^-24 of the sum of magnitudes."""
    dts = {"u8": (M.u8, M.i8, M.i32), "i8": (M.i8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.f32)}[types]
    draw = {"u8": synth.uniform_u8, "i8": synth.uniform_i8, "bf16": synth.normal_bf16}[types]
    A = draw(202, 0, (b, m, k))
    B = (synth.normal_bf16 if types == "bf16" else synth.uniform_i8)(202, 1, (b, k, n))
    C = synth.normal_f32(202, 2, (b, m, n)) if types == "bf16" else synth.uniform_i8(202, 2, (b, m, n)).astype(np.int32) * 999
    spec = M.Matmul([b, m, k, n], dts, [None, M.layout(0, 2, 1) if nk else None, None], accum)
    kernel = spec.plan().steps[-1].kernel
    as_they_lie = not nk and n % 8 != 0   # such rows go to the tile that takes them so, or are copied, by a rule of its own
    assert as_they_lie or (f"RB = {columns // 32}, SLOTS" in kernel if columns else "SLOTS" not in kernel), kernel
    got = run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, C.copy()])
    a64, b64 = _widen(A).astype(np.float64), _widen(B).astype(np.float64)
    want = a64 @ b64 + (C if accum else 0)
    if types == "bf16":
        assert (np.abs(got - want) <= (k + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + 8)).all()
    else:
        assert np.array_equal(got, want.astype(np.int32))


@pytest.mark.parametrize("types,b,m,k,n,nk,slices", [
    ("u8", 1, 65, 656, 66, True, 1),          # six steps, the last of one chunk; tiles of one row and two columns
    ("u8", 1, 193, 768, 208, False, 1),
    ("i8", 2, 80, 1040, 320, True, 1),        # entries side by side
    ("bf16", 1, 127, 328, 129, True, 1),
    ("bf16", 1, 1024, 1016, 1024, False, 1),  # a round; nine steps or more along N
    ("bf16", 3, 70, 584, 72, False, 1),
    ("bf16", 1, 33, 2696, 2051, True, 5),     # few rows
    ("u8", 1, 122, 4288, 96, False, 4),       # slices of K, the last a shorter one
    ("bf16", 1, 146, 2184, 152, False, 4),
    ("bf16", 1, 237, 2872, 203, True, 5),
])
@pytest.mark.parametrize("accum", [False, True])
@pytest.mark.parametrize("out", ["wide", "bf16"])
def test_whole_chunks_on_the_smallest_tile(gpu, types, b, m, k, n, nk, slices, accum, out):
    """As above; a bf16 result is rounded once, 2^-8 of it (half a unit of the last of eight bits)."""
    if types != "bf16" and out == "bf16":
        pytest.skip("integers stay integers")
    dts = {"u8": (M.u8, M.i8, M.i32), "i8": (M.i8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.bf16 if out == "bf16" else M.f32)}[types]
    draw = {"u8": synth.uniform_u8, "i8": synth.uniform_i8, "bf16": synth.normal_bf16}[types]
    A = draw(203, 0, (b, m, k))
    B = (synth.normal_bf16 if types == "bf16" else synth.uniform_i8)(203, 1, (b, k, n))
    if types == "bf16":
        C = (synth.normal_bf16 if out == "bf16" else synth.normal_f32)(203, 2, (b, m, n))
    else:
        C = synth.uniform_i8(203, 2, (b, m, n)).astype(np.int32) * 999
    spec = M.Matmul([b, m, k, n], dts, [None, M.layout(0, 2, 1) if nk else None, None], accum)
    plan = spec.plan()
    assert plan.kernels == ["k_gemm_ring", "k_sum_splits"][:1 + (slices > 1)] and "RA = 2, RB = 2, SLOTS" in plan.steps[0].kernel, plan
    assert slices == 1 or plan.steps[0].grid[1] == slices, plan
    got = run_spec(spec, [A, np.ascontiguousarray(B.transpose(0, 2, 1)) if nk else B, C.copy()])
    a64, b64, c64 = (_widen(x).astype(np.float64) for x in (A, B, C))
    want = a64 @ b64 + (c64 if accum else 0)
    if types == "bf16":
        slack = (k + 2 + slices) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + 8)
        assert (np.abs(_widen(got) - want) <= slack + (2.0 ** -8 * (np.abs(want) + slack) if out == "bf16" else 0)).all()
    else:
        assert np.array_equal(got, want.astype(np.int32))
