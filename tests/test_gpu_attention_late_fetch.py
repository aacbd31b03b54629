"""The fused chain while copies across PCIe keep the memory system busy: what a workgroup fetches past its last block of keys must have landed before its
halves exchange their results through the same LDS."""
import threading

import numpy as np
import pytest

import morello_amd as M
from morello_amd import synth
from gpu_util import run_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,m,k,n2", [(16, 128, 64, 512), (4, 256, 128, 512), (64, 64, 32, 256)])
@pytest.mark.parametrize("kt_rows", [True, False])
def test_results_beside_copies(gpu, b, m, k, n2, kt_rows):
    spec = M.ComposeMSM(b, m, k, n2, k, [M.bf16] * 3 + [M.f32], None if kt_rows else [None, None, M.layout(0, 2, 1), None])
    ins = [synth.normal_bf16(921, i, tuple(spec.parameter_shape(i))) for i in range(3)]
    want = run_spec(spec, ins + [np.zeros((b, m, k), np.float32)])
    # (of the one build, for the equality below: itself a softmax in float64 but for P's rounding to bf16, 2^-9 of each)
    v, q, kt = (synth.bf16_bits_to_f32(x).astype(np.float64) for x in ins)
    scores = q @ (kt if kt_rows else kt.reshape(b, n2, k).transpose(0, 2, 1))
    p = np.exp(scores - scores.max(-1, keepdims=True))
    exact = p / p.sum(-1, keepdims=True) @ v
    assert np.linalg.norm(want - exact) <= 4e-3 * np.linalg.norm(exact)
    bufs = [M.DeviceBuffer.from_numpy(x) for x in ins] + [M.DeviceBuffer(4 * b * m * k) for _ in range(20)]
    stream, stop, x = M.Stream(), threading.Event(), np.ones(1 << 20, np.float32)

    def copies():
        out = np.zeros_like(x)
        while not stop.is_set():
            M.Move([x.size], (M.f32, M.f32)).run_host(x, out)

    threads = [threading.Thread(target=copies) for _ in range(2)]
    for t in threads:
        t.start()
    try:
        for _ in range(5):
            for out in bufs[3:]:
                spec.run_async([v.ptr for v in bufs[:3]] + [out.ptr], stream)
            stream.synchronize()
            for out in bufs[3:]:
                assert np.array_equal(out.to_numpy(np.float32, want.shape), want)
    finally:
        stop.set()
        for t in threads:
            t.join()
    for v in bufs:
        v.free()
    stream.destroy()
