"""The row factors of the matrix-core last pass (2^18..2^22 and 2^24): transforms
whose tables came with ntt_set_up or with a larger transform, under capture, after
the field's own tables are gone, and on a GPU too full for them."""
import ctypes

import numpy as np
import pytest

import bellman_amd as B
from gpu_helpers import ntt

pytestmark = pytest.mark.gpu


def fresh_tables():
    B.call("ntt_tear_down")
    B.call("ntt_set_up")


def free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    B.call("bc_mem_get_info", ctypes.byref(free), ctypes.byref(total))
    return free.value, total.value


@pytest.mark.parametrize("log_n", [18, 20])
@pytest.mark.parametrize("inverse", [False, True])
def test_first_use_under_capture(bellman, oracle, log_n, inverse):
    _, dev = bellman
    fresh_tables()
    hip = B.lib()  # finds the HIP functions it is linked with
    xs = [oracle.random_fr(0xBC0000E7 + i, 1 << log_n) for i in range(3)]
    d_in, d_out = dev.malloc(32 << log_n), dev.malloc(32 << log_n)
    cfg = B.ntt_configuration()
    cfg.mem_pool, cfg.stream, cfg.inputs, cfg.outputs, cfg.log_values_count, cfg.inverse = dev.pool, dev.stream, d_in, d_out, log_n, inverse
    graph, instance = ctypes.c_void_p(), ctypes.c_void_p()
    stream = ctypes.c_void_p(dev.stream.handle)
    assert hip.hipStreamBeginCapture(stream, ctypes.c_int(2)) == 0  # hipStreamCaptureModeRelaxed
    B.call("ntt_execute_async", cfg)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(instance), graph, None, None, ctypes.c_size_t(0)) == 0
    for x in xs:
        B.call("bc_memcpy", ctypes.c_void_p(d_in), B.ptr(x), ctypes.c_size_t(x.nbytes))
        assert hip.hipGraphLaunch(instance, stream) == 0
        dev.sync()
        want = oracle.ntt(x, log_n, False, inverse)
        assert np.array_equal(dev.download(d_out, (1 << log_n, 8)), want)
        assert np.array_equal(ntt(dev, x, log_n, inverse=inverse), want)
    assert hip.hipGraphExecDestroy(instance) == 0
    assert hip.hipGraphDestroy(graph) == 0
    dev.free(d_in)
    dev.free(d_out)


def test_transforms_outlive_the_field_tables(bellman, oracle):
    _, dev = bellman
    fresh_tables()
    B.call("ff_tear_down")
    try:
        for log_n in (10, 18, 20):
            x = oracle.random_fr(0xBC0000F7 + log_n, 1 << log_n)
            for inverse in (False, True):
                assert np.array_equal(ntt(dev, x, log_n, inverse=inverse), oracle.ntt(x, log_n, False, inverse))
    finally:
        B.call("ff_set_up", ctypes.c_uint(25), ctypes.c_uint(14))
        B.call("pn_set_up")


def test_transforms_without_the_tables(bellman, oracle):
    """All but 16 GiB of the GPU's memory taken, below the eighth that the tables
    leave alone: two or three matrix-core passes are followed by a VALU pass of 6..10
    stages.  With the memory back, the same inputs on the last pass."""
    _, dev = bellman
    B.call("ntt_tear_down")
    free, total = free_memory()
    held = []
    inputs = {}
    try:
        while free_memory()[0] > 20 << 30:
            p = ctypes.c_void_p()
            B.call("bc_malloc", ctypes.byref(p), ctypes.c_size_t(min(32 << 30, free_memory()[0] - (16 << 30))))
            held.append(p)
        before = free_memory()[0]
        assert before < total // 8
        B.call("ntt_set_up")
        assert before - free_memory()[0] < 32 * (2 << 20) + (32 << 20)  # the twiddles to 2^20, no more
        for log_n in (18, 19, 20, 21, 22, 24):
            x = oracle.random_fr(0xBC0000F8 + log_n, 1 << log_n)
            x[3::13] = oracle.to_limbs([oracle.R - 1])[0]
            for inverse, log_ext in [(False, 0)] if log_n == 24 else [(False, 0), (True, 0), (False, 1), (True, 1)]:
                want = oracle.ntt(x, log_n, False, inverse, log_ext, log_ext)
                assert np.array_equal(ntt(dev, x, log_n, inverse=inverse, log_ext=log_ext, coset=log_ext), want), (log_n, inverse, log_ext)
                if log_ext == 0 and not inverse:
                    inputs[log_n] = x, want
    finally:
        for p in held:
            B.call("bc_free", p)
        fresh_tables()
    for log_n, (x, want) in inputs.items():
        assert np.array_equal(ntt(dev, x, log_n), want), log_n
