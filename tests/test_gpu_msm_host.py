"""Host scalars of msm_execute_async around the sizes where the copy is split:
one copy on the call's stream below 2^20, chunks on a copy stream from there on,
for a created stream and for the null stream, which created streams wait for."""
import ctypes

import numpy as np
import pytest

from gpu_helpers import CopyHooks, msm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [4, 18, 20])
@pytest.mark.parametrize("null_stream", [False, True])
def test_pinned_scalars_on_either_stream(bellman, oracle, log_n, null_stream):
    B, dev = bellman
    n = 1 << log_n
    bases = oracle.gen_bases_progression(0xBC0000A1, 12345, n)
    k = oracle.msm_scalars(0xBC0000A2, n)
    db = dev.upload(bases)
    want = msm(dev, db, k, log_n)
    pinned = ctypes.c_void_p()
    B.call("bc_malloc_host", ctypes.byref(pinned), ctypes.c_size_t(k.nbytes))
    hooks = CopyHooks()
    d_r = dev.malloc(254 * 96)
    try:
        ctypes.memmove(pinned, k.ctypes.data, k.nbytes)
        cfg = B.msm_configuration()
        cfg.mem_pool, cfg.stream = dev.pool, B.bc_stream() if null_stream else dev.stream
        cfg.bases, cfg.scalars, cfg.results, cfg.log_scalars_count = db, pinned.value, d_r, log_n
        hooks.attach(cfg)
        B.call("msm_execute_async", cfg)
        B.call("bc_stream_synchronize", cfg.stream)
        got = dev.download(d_r, (254, 24))
        assert np.array_equal(oracle.to_affine(got), oracle.to_affine(want))
        assert hooks.wait_calls(1) == [CopyHooks.H2D]
        assert hooks.events_complete()
    finally:
        hooks.close()
        B.call("bc_free_host", pinned)
        dev.free(d_r)
        dev.free(db)
