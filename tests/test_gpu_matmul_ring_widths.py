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
    ("bf16", 1, 1153, 832, 832, 0),        # 247 tiles
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
