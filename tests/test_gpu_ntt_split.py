"""A named first pass where the passes follow it: launches of more than 2^17
elements of sizes below 2^18, and bit-reversed inputs from there on."""
import ctypes

import numpy as np
import pytest

from gpu_helpers import ntt, ntt_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [7, 8, 10])
def test_two_transforms_of_2_17(bellman, oracle, split):
    B, dev = bellman
    log_n, first = 17, ctypes.c_uint()
    B.call("bc_amd_ntt_get_split", ctypes.c_uint(log_n), ctypes.byref(first))
    B.call("bc_amd_ntt_set_split", ctypes.c_uint(log_n), ctypes.c_uint(split))
    try:
        for bitrev in (False, True):
            xs = [oracle.random_fr(0xBC0000FC + i, 1 << log_n) for i in range(2)]
            bufs = [dev.upload(x) for x in xs]
            ntt_batch(dev, [B.ntt_job(p, p, log_n, bitrev=bitrev, inverse=i == 1) for i, p in enumerate(bufs)])
            for i, (p, x) in enumerate(zip(bufs, xs)):
                assert np.array_equal(dev.download(p, (1 << log_n, 8)), oracle.ntt(x, log_n, bitrev, i == 1)), (bitrev, i)
                dev.free(p)
    finally:
        B.call("bc_amd_ntt_set_split", ctypes.c_uint(log_n), first)


@pytest.mark.parametrize("log_n,splits", [(18, (8, 10)), (20, (10,)), (22, (2, 10))])
def test_bit_reversed_inputs(bellman, oracle, log_n, splits):
    B, dev = bellman
    first = ctypes.c_uint()
    x = oracle.random_fr(0xBC0000FE + log_n, 1 << log_n)
    B.call("bc_amd_ntt_get_split", ctypes.c_uint(log_n), ctypes.byref(first))
    try:
        for inverse in (False, True):
            want = oracle.ntt(x, log_n, True, inverse)
            for split in splits:
                B.call("bc_amd_ntt_set_split", ctypes.c_uint(log_n), ctypes.c_uint(split))
                assert np.array_equal(ntt(dev, x, log_n, bitrev=True, inverse=inverse), want), (inverse, split)
    finally:
        B.call("bc_amd_ntt_set_split", ctypes.c_uint(log_n), first)
