"""Fr vector operations at the edges of their kernels' tiles and chunks, against
the CPU oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one block up to 256 (an element a thread) and 1024, tiles of 1024 up to 2^20, chunks of 8 in tiles above
@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2048, 2049, 200001, 1 << 20, (1 << 20) + 1, (1 << 20) + 8199])
@pytest.mark.parametrize("in_place", [False, True])
def test_grand_product_at_tile_edges(bellman, oracle, n, in_place):
    B, dev = bellman
    x = oracle.random_fr(n + 11, n)
    dx = dev.upload(x)
    dy = dx if in_place else dev.malloc(n * 32)
    B.call("ff_grand_product", B.ff_grand_product_configuration(dev.pool, dev.stream, dx, dy, n))
    dev.sync()
    assert np.array_equal(dev.download(dy, (n, 8)), oracle.grand_product(x))
    dev.free(dx)
    if not in_place:
        dev.free(dy)


# a power per thread up to 2^17 elements, the two tables above; one evaluation
# block up to 2048; tiles of 512 up to 2^17, 2048 up to 2^21, 8192 above, then one block
@pytest.mark.parametrize("n", [0, 1, 2, 64, 65, 255, 256, 257, 511, 513, 2049, 65539, 1 << 17, (1 << 17) + 1, (1 << 20) + 3, (1 << 21) + 1])
@pytest.mark.parametrize("on_device", [False, True])
def test_powers_and_evaluation_at_tile_edges(bellman, oracle, n, on_device):
    B, dev = bellman
    x = oracle.random_fr(n + 13, max(n, 1))
    base = oracle.random_fr(n + 17, 1)
    dx, dy, db, dr = dev.upload(x), dev.malloc(max(n, 1) * 32), dev.upload(base), dev.malloc(32)
    result = np.zeros((1, 8), dtype=np.uint32)
    B.call("ff_poly_evaluate", B.ff_poly_evaluate_configuration(dev.pool, dev.stream, dx, db if on_device else base.ctypes.data,
                                                                dr if on_device else result.ctypes.data, n))
    B.call("ff_multiply_by_powers", B.ff_multiply_by_powers_configuration(dev.pool, dev.stream, dx, db if on_device else base.ctypes.data, dy, n))
    dev.sync()
    if on_device:
        result = dev.download(dr, (1, 8))
    assert np.array_equal(result, oracle.poly_evaluate(x[:n], base) if n else np.zeros((1, 8), dtype=np.uint32))
    if n:
        expected = oracle.multiply_by_powers(x, base)
        assert np.array_equal(dev.download(dy, (n, 8)), expected)
        B.call("ff_multiply_by_powers", B.ff_multiply_by_powers_configuration(dev.pool, dev.stream, dx, db if on_device else base.ctypes.data, dx, n))
        dev.sync()
        assert np.array_equal(dev.download(dx, (n, 8)), expected)
    for p in (dx, dy, db, dr):
        dev.free(p)


@pytest.mark.parametrize("point", [0, 1, -1])
def test_evaluation_at_special_points(bellman, oracle, point):
    B, dev = bellman
    n = 5001
    x = oracle.random_fr(19, n)
    base = oracle.to_mont([point % oracle.R])
    dx = dev.upload(x)
    result = np.zeros((1, 8), dtype=np.uint32)
    B.call("ff_poly_evaluate", B.ff_poly_evaluate_configuration(dev.pool, dev.stream, dx, base.ctypes.data, result.ctypes.data, n))
    dev.sync()
    assert np.array_equal(result, oracle.poly_evaluate(x, base))
    dev.free(dx)


# one thread an element below 2^8, then tiles of 256: a single one, one with no
# middle bit to reverse, odd and even numbers of middle bits
@pytest.mark.parametrize("log_n", [2, 7, 8, 9, 10, 11, 15, 18])
def test_bit_reverse_at_tile_edges(bellman, oracle, log_n):
    B, dev = bellman
    n = 1 << log_n
    x = oracle.random_fr(log_n + 29, n)
    dx, dy = dev.upload(x), dev.malloc(n * 32)
    for src, dst in ((dx, dy), (dx, dx)):
        B.call("ff_bit_reverse", ctypes.c_void_p(src), ctypes.c_void_p(dst), ctypes.c_uint(log_n), dev.stream)
        dev.sync()
        assert np.array_equal(dev.download(dst, (n, 8)), oracle.bit_reverse(x, log_n))
    dev.free(dx)
    dev.free(dy)
