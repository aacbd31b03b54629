"""Row-major right operands copied in panels as wide as the tile that reads them (gemm_ring.hip), against float64."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu


def _widen(x):
    return (x.astype(np.uint32) << 16).view(np.float32) if x.dtype == np.uint16 else x


@pytest.mark.parametrize("types,b,m,k,n,columns", [
    ("u8", 1, 1408, 3203, 1409, 64),     # the last panel one column wide
    ("u8", 1, 1408, 3201, 1471, 64),     # ... one short of whole; K a byte past whole chunks
    ("u8", 2, 700, 3001, 2881, 160),     # two entries
    ("u8", 1, 1793, 3999, 3009, 192),
    ("bf16", 1, 1930, 2111, 1921, 128),
    ("bf16", 1, 1001, 2311, 4321, 160),
    ("bf16", 2, 643, 2307, 2911, 160),
    ("bf16", 1, 1793, 2503, 3071, 192),
    ("bf16", 1, 1100, 4000, 1101, 64),   # only B is copied
])
@pytest.mark.parametrize("accum", [False, True])
def test_panels(gpu, types, b, m, k, n, columns, accum):
    """Integers exact; bf16 sums of k products in f32 are within k rounding errors of 2^-24 of the sum of magnitudes."""
    dts = {"u8": (M.u8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.f32)}[types]
    A = (synth.uniform_u8 if types == "u8" else synth.normal_bf16)(201, 0, (b, m, k))
    B = (synth.uniform_i8 if types == "u8" else synth.normal_bf16)(201, 1, (b, k, n))
    C = synth.uniform_i8(201, 2, (b, m, n)).astype(np.int32) * 999 if types == "u8" else synth.normal_f32(201, 2, (b, m, n))
    spec = M.Matmul([b, m, k, n], dts, accum=accum)
    plan = spec.plan()
    assert plan.kernels[0] in ("k_pad_rows", "k_pad_rows_pair") and f"RB = {columns // 32}, SLOTS" in plan.steps[-1].kernel, plan
    got = run_spec(spec, [A, B, C.copy()])
    a64, b64 = _widen(A).astype(np.float64), _widen(B).astype(np.float64)
    want = a64 @ b64 + (C if accum else 0)
    if types == "u8":
        assert np.array_equal(got, want.astype(np.int32))
    else:
        assert (np.abs(got - want) <= (k + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + 8)).all()
