"""Matrix-vector products with one and with two rows of B per wavefront (gemv.hip), on either side of 80 and 200 MB of B."""
import numpy as np
import pytest

import morello_amd as M
from gpu_util import run_spec
from morello_amd import synth

pytestmark = pytest.mark.gpu

KT = M.layout(0, 2, 1)


@pytest.mark.parametrize("m,k,n", [(1, 4112, 11003), (2, 4112, 11003), (1, 2064, 38001), (2, 2064, 38001), (1, 12304, 6701), (2, 12304, 6701), (1, 16384, 12209)])
def test_rows_of_b_per_wavefront(gpu, m, k, n):
    """Whole numbers bit for bit; a ragged last chunk of K and a column count of no whole workgroups."""
    a, b = synth.uniform_u8(195, 0, (1, m, k)), synth.uniform_i8(195, 1, (1, n, k))
    spec = M.Matmul([1, m, k, n], (M.u8, M.i8, M.i32), layouts=[None, KT, None])
    assert spec.plan().kernels == ["k_gemv"]
    got = run_spec(spec, [a, b, np.full((1, m, n), 7, np.int32)])
    want = np.concatenate([a[0].astype(np.float64) @ b[0, i:i + 1000].astype(np.float64).T for i in range(0, n, 1000)], 1)   # (below 2^53: exact)
    assert np.array_equal(got[0].astype(np.float64), want)
