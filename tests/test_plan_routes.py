"""Which kernels a Spec goes to where two routes meet, by its plan (no GPU): Specs that one of them cannot
take, or takes at many times the other's cost."""
import pytest

import morello_amd as M

KT = M.layout(0, 2, 1)


@pytest.mark.parametrize("batch,k", [(1 << 27, 1), ((1 << 27) + 1, 3)])
def test_operands_too_many_for_padded_copies_stay_as_they_are(batch, k):
    """2^27 right operands of up to 16 rows of a chunk each are 2^31 chunks, more than the copy numbers."""
    p = M.Matmul([batch, 1, k, 1], (M.u8, M.i8, M.i32)).plan()
    assert p.kernels[-1] == "k_matmul_generic"
