"""Specs called on host buffers (mrl_run_host) through the pinned stage that stays between calls:
transfers of one part and of many (more parts than the stage has slots), parameters that are read,
read and written, and only written, stages shared out among threads, and given back."""
import ctypes as C
import threading

import numpy as np
import pytest

import morello_amd as M
import morello_amd._binding as B
import orc
from morello_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 131072 // 4, 131072 // 4 + 1, 1 << 19, (1 << 20) + 5, 9 * (1 << 20) + 3, 20 * (1 << 20) + 1])
def test_copies_of_every_length(gpu, n):
    """A Move copies its input: parts of 128 KiB and of 2 MiB, a last part of a few bytes, and (80 MB) a
    slot used three times over."""
    x = synth.uniform_f32(901, n % 7, (n,))
    out = np.zeros(n, np.float32)
    M.Move([n], (M.f32, M.f32)).run_host(x, out)
    assert np.array_equal(x, out)


@pytest.mark.parametrize("m,k,n", [(5, 64, 7), (300, 500, 700), (1024, 2048, 1536)])
def test_accumulating_output_goes_both_ways(gpu, m, k, n):
    a, b = synth.uniform_u8(902, 0, (1, m, k)), synth.uniform_i8(902, 1, (1, k, n))
    c = np.arange(m * n, dtype=np.int32).reshape(1, m, n)
    want = orc.matmul([1, m, k, n], [0, 1, 5], a, b, c.copy(), True)
    M.MatmulAccum([1, m, k, n], (M.u8, M.i8, M.i32)).run_host(a, b, c)
    assert np.array_equal(c, want)


def test_two_outputs_and_none_read(gpu):
    x = synth.normal_f32(903, 0, (64, 300), 2.0)
    mx, den = np.zeros((64, 1), np.float32), np.zeros((64, 1), np.float32)
    M.SoftmaxDenominatorAndMax([64, 300], 1).run_host(x, mx, den)
    assert np.array_equal(mx[:, 0], x.max(axis=1))
    assert np.allclose(den[:, 0], np.exp(x.astype(np.float64) - mx).sum(axis=1), rtol=1e-5)
    z = np.ones(1000, np.float32)
    M.Fill([1000], M.f32, M.FillValue.Zero).run_host(z)
    assert not z.any()


def test_threads_use_a_stage_each_and_stages_are_given_back(gpu):
    n = 3 * (1 << 20) + 17
    bad = []

    def work(t):
        x = synth.uniform_f32(904, t, (n,))
        for _ in range(3):
            out = np.zeros(n, np.float32)
            M.Move([n], (M.f32, M.f32)).run_host(x, out)
            if not np.array_equal(x, out):
                bad.append(t)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    free = []
    for _ in range(4):   # (the runtime itself may keep what the first rounds freed)
        work(0)
        M.release_stream()
        free.append(M.device_free_bytes())
    assert free[-1] >= free[1] and not bad


@pytest.mark.parametrize("on_stream", [False, True])
def test_host_buffers_that_earlier_work_still_fills(gpu, on_stream):
    """The call comes behind what the null stream, and a stream that synchronises with it, hold: an input in
    pinned memory that a Move writes behind some milliseconds of Matmul."""
    n = 1 << 20
    hip, pin = B.load(), C.c_void_p()
    hip.hipHostMalloc.argtypes, hip.hipHostFree.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint], [C.c_void_p]
    assert hip.hipHostMalloc(C.byref(pin), 4 * n, 0) == 0
    x, out = np.ctypeslib.as_array(C.cast(pin, C.POINTER(C.c_float)), (n,)), np.zeros(n, np.float32)
    long_one, move = M.Matmul([1, 8192, 8192, 8192], (M.f32, M.f32, M.f32)), M.Move([n], (M.f32, M.f32))
    bufs = [M.DeviceBuffer(4 << 26) for _ in range(3)]
    stream = M.Stream() if on_stream else None
    enqueue = (lambda spec, ptrs: spec.run_async(ptrs, stream)) if on_stream else (lambda spec, ptrs: spec.run_noalloc(ptrs))
    for value in (3.0, 4.0):
        src = M.DeviceBuffer.from_numpy(np.full(n, value, np.float32))
        x[:] = -1.0
        M.synchronize()
        enqueue(long_one, [b.ptr for b in bufs])
        enqueue(move, [src.ptr, pin.value])
        move.run_host(x, out)
        assert (out == value).all()
        M.synchronize()
        src.free()
    for b in bufs:
        b.free()
    if stream:
        stream.destroy()
    hip.hipHostFree(pin)
