"""The fused Matmul -> Softmax -> Matmul on head dims of whole 16-byte chunks that it reads in place (k_attn with
NARROW), against float64 on the CPU."""
import numpy as np
import pytest

import morello_amd as M
from gpu_util import run_spec
from morello_amd import synth

pytestmark = pytest.mark.gpu
KT = M.layout(0, 2, 1)


def _f64(bits):
    return synth.bf16_bits_to_f32(bits).astype(np.float64)


def _want(v, q, k):
    s = _f64(q) @ _f64(k).transpose(0, 2, 1)
    with np.errstate(invalid="ignore"):
        p = np.exp(s - s.max(-1, keepdims=True))
    return p / p.sum(-1, keepdims=True) @ _f64(v)


@pytest.mark.parametrize("k,n", [(80, 80), (96, 96), (96, 72), (128, 40), (8, 120), (40, 48), (64, 56), (48, 128)])
@pytest.mark.parametrize("b,m,keys", [(3, 100, 321), (2, 257, 64), (40, 130, 1000), (2, 1, 5000), (1, 33, 7)])
def test_head_dims_read_in_place(gpu, b, m, keys, k, n):
    """Query and key counts on either side of the blocks of 32, 64 and 128, one and both halves of the keys, keys shared
    out over workgroups.  The probabilities are rounded to bf16 (2^-9 of each), as for the whole head dims: 1e-2 in the norm."""
    v, q, kk = (synth.normal_bf16(180, i, s, 0.5) for i, s in enumerate([(b, keys, n), (b, m, k), (b, keys, k)]))
    spec = M.ComposeMSM(b, m, k, keys, n, layouts=[None, None, KT, None])
    steps = spec.plan().steps
    assert spec.plan().kernels[0] == "k_attn" and "NARROW = true" in steps[0].kernel
    got = run_spec(spec, [v, q, kk, np.full((b, m, n), 7, np.float32)]).astype(np.float64)
    want = _want(v, q, kk)
    assert np.linalg.norm(got - want) <= 1e-2 * np.linalg.norm(want)


def test_a_row_of_keys_does_not_reach_into_its_neighbour(gpu):
    """An infinity at the start of a row lies where the row before it, taken as 128 elements long, would end: a key whose
    score is -inf drops out, and no other key's score holds it; likewise past the last query and the last key."""
    b, m, keys, d = 2, 70, 130, 80
    v, q, kk = (synth.normal_bf16(181, i, s, 0.5) for i, s in enumerate([(b, keys, d), (b, m, d), (b, keys, d)]))
    q[:, :, 0] = 0x3f80           # 1
    kk[:, 5::9, 0] = 0xff80       # -inf
    spec = M.ComposeMSM(b, m, d, keys, d, layouts=[None, None, KT, None])
    got = run_spec(spec, [v, q, kk, np.zeros((b, m, d), np.float32)])
    want = _want(v, q, kk)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert np.linalg.norm(got - want) <= 1e-2 * np.linalg.norm(want)
