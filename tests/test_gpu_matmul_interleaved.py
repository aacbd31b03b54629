"""Row-major right operands whose batch entries' rows lie between each other ([k][batch][n] in memory), read in place by the tiles that
work on whole 16-byte chunks, against float64: the last row of the last entry is the operand's end, wherever the tile's columns end."""
import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu
TYPES = {"u8": (M.u8, M.i8, M.i32), "i8": (M.i8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.f32), "f32": (M.f32, M.f32, M.f32)}
DRAW = {M.u8: synth.uniform_u8, M.i8: synth.uniform_i8, M.bf16: synth.normal_bf16, M.f32: synth.normal_f32}


def _widen(x):
    return (x.astype(np.uint32) << 16).view(np.float32) if x.dtype == np.uint16 else x


@pytest.mark.parametrize("types,b,m,k,n,kernel,tile", [
    ("bf16", 2, 70, 1024, 72, "k_gemm_ring", "RA = 2, RB = 2"),     # 64 x 64: the last column of tiles 8 wide
    ("u8", 3, 96, 1536, 80, "k_gemm_ring", "RA = 2, RB = 2"),
    ("u8", 2, 130, 4104, 208, "k_gemm_ring", "RA = 2, RB = 2"),     # K ends within a step
    ("bf16", 2, 1153, 776, 456, "k_gemm_ring", "RA = 4, RB = 2"),
    ("bf16", 2, 1000, 1792, 1160, "k_gemm_ring", "RA = 4, RB = 4"),
    ("u8", 2, 700, 3008, 2896, "k_gemm_ring", "RA = 4, RB = 5"),
    ("bf16", 2, 900, 2312, 3064, "k_gemm_ring", "RA = 4, RB = 6"),
    ("bf16", 2, 422, 448, 880, "k_gemm", "Tile<64, 64"),
    ("u8", 2, 1000, 1024, 1104, "k_gemm", "Tile<128, 128"),
    ("bf16", 2, 1000, 520, 1104, "k_gemm", "Tile<128, 128"),
    ("bf16", 2, 2040, 512, 2056, "k_gemm", "Tile<256, 256"),
    ("f32", 3, 70, 64, 72, "k_gemm", "Tile<64, 64"),
])
@pytest.mark.parametrize("accum", [False, True])
def test_entries_between_each_other(gpu, types, b, m, k, n, kernel, tile, accum):
    """Integers exact; sums of k products in f32 are within k rounding errors of 2^-24 of the sum of magnitudes."""
    dts = TYPES[types]
    A, B = DRAW[dts[0]](211, 0, (b, m, k)), DRAW[dts[1]](211, 1, (b, k, n))
    C = synth.normal_f32(211, 2, (b, m, n)) if dts[2] == M.f32 else synth.uniform_i8(211, 2, (b, m, n)).astype(np.int32) * 999
    spec = M.Matmul([b, m, k, n], dts, [None, M.layout(1, 0, 2), None], accum)
    steps = spec.plan().steps
    assert len(steps) == 1 and steps[0].kernel.split()[0] == kernel and tile in steps[0].kernel, steps
    got = run_spec(spec, [A, np.ascontiguousarray(B.transpose(1, 0, 2)), C.copy()])
    a64, b64 = _widen(A).astype(np.float64), _widen(B).astype(np.float64)
    want = a64 @ b64 + (C if accum else 0)
    if dts[2] == M.f32:
        assert (np.abs(got - want) <= (k + 2) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + 8)).all()
    else:
        assert np.array_equal(got, want.astype(np.int32))
