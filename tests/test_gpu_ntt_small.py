"""Transforms of launches that cannot fill the GPU (up to 2^17 elements in all):
every size, order and direction around their tiles of 512 elements, alone, on
cosets and batched on both sides of that line."""
import numpy as np
import pytest

from gpu_helpers import ntt, ntt_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [1, 2, 3, 4, 6, 7, 8, 9, 10, 11, 14, 15, 17])
@pytest.mark.parametrize("bitrev", [False, True])
@pytest.mark.parametrize("inverse", [False, True])
def test_small_transforms(bellman, oracle, log_n, bitrev, inverse):
    _, dev = bellman
    x = oracle.random_fr(0xBC0000C1 + log_n, 1 << log_n)
    x[::3] = oracle.to_limbs([oracle.R - 1])[0]
    assert np.array_equal(ntt(dev, x, log_n, bitrev=bitrev, inverse=inverse), oracle.ntt(x, log_n, bitrev, inverse))
    assert np.array_equal(ntt(dev, x, log_n, bitrev=bitrev, inverse=inverse, log_ext=1, coset=1), oracle.ntt(x, log_n, bitrev, inverse, 1, 1))


@pytest.mark.parametrize("logs", [[16, 15, 15, 9], [16, 16], [16, 16, 1], [10, 3, 12, 16, 7]])
def test_batches_around_the_line(bellman, oracle, logs):
    B, dev = bellman
    xs = [oracle.random_fr(0xBC0000D1 + i, 1 << l) for i, l in enumerate(logs)]
    bufs = [dev.upload(x) for x in xs]
    ntt_batch(dev, [B.ntt_job(p, p, l, bitrev=i % 2 == 1, inverse=i % 3 == 1, log_ext=i % 2, coset=0) for i, (p, l) in enumerate(zip(bufs, logs))])
    for i, (p, x, l) in enumerate(zip(bufs, xs, logs)):
        assert np.array_equal(dev.download(p, (1 << l, 8)), oracle.ntt(x, l, i % 2 == 1, i % 3 == 1, i % 2, 0)), i
        dev.free(p)


@pytest.mark.parametrize("split", [6, 7, 10])
def test_named_first_pass_in_a_larger_launch(bellman, oracle, split):
    """A first pass named for a size serves launches above the line, both orders."""
    import ctypes

    B, dev = bellman
    log_n, first = 16, ctypes.c_uint()
    xs = [oracle.random_fr(0xBC0000E1 + i, 1 << log_n) for i in range(3)]
    B.call("bc_amd_ntt_get_split", ctypes.c_uint(log_n), ctypes.byref(first))
    B.call("bc_amd_ntt_set_split", ctypes.c_uint(log_n), ctypes.c_uint(split))
    try:
        bufs = [dev.upload(x) for x in xs]
        ntt_batch(dev, [B.ntt_job(p, p, log_n, bitrev=i == 1, inverse=i == 2) for i, p in enumerate(bufs)])
        for i, (p, x) in enumerate(zip(bufs, xs)):
            assert np.array_equal(dev.download(p, (1 << log_n, 8)), oracle.ntt(x, log_n, i == 1, i == 2)), i
            dev.free(p)
        assert np.array_equal(ntt(dev, xs[0], log_n), oracle.ntt(xs[0], log_n))
    finally:
        B.call("bc_amd_ntt_set_split", ctypes.c_uint(log_n), first)
