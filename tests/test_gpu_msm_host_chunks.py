"""Pinned host inputs of msm_execute_async at 2^22 points, the smallest size that
is copied in four chunks: each of the two staging slots is used twice."""
import ctypes

import numpy as np
import pytest

from gpu_helpers import CopyHooks, msm

pytestmark = pytest.mark.gpu
LOG_N = 22


@pytest.fixture(scope="module")
def inputs(bellman, oracle):
    """Bases (multiples of the generator), scalars, and the per-bit results from device memory."""
    B, dev = bellman
    n = 1 << LOG_N
    s = np.random.default_rng(0xBC0000FA).integers(0, 1 << 32, size=(n, 8), dtype=np.uint32)
    s[:, 7] %= 0x30644E72  # below r's top word
    k = oracle.msm_scalars(0xBC0000FB, n)
    d_s, d_b = dev.upload(s), dev.malloc(64 * n)
    B.call("bc_amd_generator_multiples", ctypes.c_void_p(d_s), ctypes.c_void_p(d_b), ctypes.c_uint(n), dev.stream)
    dev.sync()
    dev.free(d_s)
    want = oracle.to_affine(msm(dev, d_b, k, LOG_N))
    yield d_b, k, want
    dev.free(d_b)


@pytest.mark.parametrize("pinned_bases,pinned_scalars", [(False, True), (True, False), (True, True)])
@pytest.mark.parametrize("null_stream", [False, True])
def test_four_chunks(bellman, oracle, inputs, pinned_bases, pinned_scalars, null_stream):
    B, dev = bellman
    d_b, k, want = inputs
    d_k, d_r = dev.upload(k), dev.malloc(254 * 96)
    hooks = CopyHooks()
    held = []

    def address(device, nbytes, pinned):
        if not pinned:
            return device
        p = ctypes.c_void_p()
        B.call("bc_malloc_host", ctypes.byref(p), ctypes.c_size_t(nbytes))
        held.append(p)
        B.call("bc_memcpy", p, ctypes.c_void_p(device), ctypes.c_size_t(nbytes))
        return p.value

    try:
        cfg = B.msm_configuration()
        cfg.mem_pool, cfg.stream = dev.pool, B.bc_stream() if null_stream else dev.stream
        cfg.bases, cfg.scalars = address(d_b, 64 << LOG_N, pinned_bases), address(d_k, 32 << LOG_N, pinned_scalars)
        cfg.results, cfg.log_scalars_count = d_r, LOG_N
        hooks.attach(cfg)
        for _ in range(2):  # the second call finds the first one's staging memory in the pool
            B.call("bc_memset", ctypes.c_void_p(d_r), ctypes.c_int(0x5A), ctypes.c_size_t(254 * 96))
            B.call("msm_execute_async", cfg)
            B.call("bc_stream_synchronize", cfg.stream)
            assert np.array_equal(oracle.to_affine(dev.download(d_r, (254, 24))), want)
        assert hooks.wait_calls(2) == [CopyHooks.H2D] * 2
        assert hooks.events_complete()
    finally:
        hooks.close()
        for p in held:
            B.call("bc_free_host", p)
        dev.free(d_k)
        dev.free(d_r)
