"""The cost model beside launches measured on an MI355X, back to back on one set of operands.  No GPU needed."""
import pytest

import morello_amd as M

KT = M.layout(0, 2, 1)


@pytest.mark.parametrize("types,b,m,k,n,nk,us", [
    ("bf16", 1, 1024, 1024, 1024, False, 6.7), ("u8", 1, 512, 1024, 512, True, 4.9), ("bf16", 2, 86, 2144, 264, True, 7.5),
    ("u8", 2, 615, 5760, 112, False, 12.8), ("u8", 1, 693, 4352, 816, True, 11.5), ("bf16", 1, 384, 512, 768, True, 4.3),
])
def test_small_matmuls(types, b, m, k, n, nk, us):
    """One launch of 64 x 64 tiles fed straight into LDS, whose chain of steps sets its time: within a quarter."""
    p = M.Matmul([b, m, k, n], (M.u8, M.i8, M.i32) if types == "u8" else (M.bf16, M.bf16, M.f32), [None, KT if nk else None, None]).plan()
    assert p.kernels == ["k_gemm_ring"] and "RA = 2, RB = 2, SLOTS" in p.steps[0].kernel, p
    assert abs(p.cost_ns - 1e3 * us) <= 0.25 * 1e3 * us, p


@pytest.mark.parametrize("types,b,c,f,hw,fs,us", [("bf16", 21, 144, 64, 17, 3, 6.7), ("u8", 1, 64, 48, 21, 5, 5.7), ("bf16", 2, 96, 48, 69, 3, 5.9), ("u8", 6, 96, 128, 20, 3, 5.2)])
def test_small_convs(types, b, c, f, hw, fs, us):
    p = M.Conv([b, f, c, hw, hw, fs, fs], (M.u8, M.i8, M.i32) if types == "u8" else (M.bf16, M.bf16, M.f32)).plan()
    assert p.kernels == ["k_gemm"] and "RA = 2" in p.steps[0].kernel, p
    assert abs(p.cost_ns - 1e3 * us) <= 0.25 * 1e3 * us, p
