"""Inputs that are not reduced: values of the field stored with multiples of r
added.  Results are those of the reduced values."""
import numpy as np
import pytest

from gpu_helpers import ntt

pytestmark = pytest.mark.gpu


def add_multiples(oracle, x, most):
    """Element i of x plus i % (most + 1) times r, or as much of that as 256 bits hold."""
    out = x.astype(np.uint64)
    r = oracle.to_limbs([oracle.R])[0].astype(np.uint64)
    k = np.arange(len(x), dtype=np.uint64) % np.uint64(most + 1)
    if most > 4:  # 6 r > 2^256 > 5 r: the small elements alone hold five
        k[(k == 5) & (x[:, 7] >= 0x0D000000)] = 4
    carry = np.zeros(len(x), dtype=np.uint64)
    for i in range(8):
        s = out[:, i] + k * r[i] + carry
        out[:, i], carry = s & np.uint64(0xFFFFFFFF), s >> np.uint64(32)
    assert not carry.any()
    return out.astype(np.uint32)


@pytest.mark.parametrize("log_n", [9, 12, 17, 18, 20, 23])
@pytest.mark.parametrize("inverse,log_ext", [(False, 0), (True, 0), (False, 1)])
def test_natural_order_transforms_below_4r(bellman, oracle, log_n, inverse, log_ext):
    _, dev = bellman
    x = oracle.random_fr(0xBC0000A7 + log_n, 1 << log_n)
    x[::5] = oracle.to_limbs([oracle.R - 1])[0]
    got = ntt(dev, add_multiples(oracle, x, 3), log_n, inverse=inverse, log_ext=log_ext, coset=log_ext)
    assert np.array_equal(got, oracle.ntt(x, log_n, False, inverse, log_ext, log_ext))


@pytest.mark.parametrize("log_n", [9, 12, 17, 18, 20, 23])
def test_forward_coset_transforms_of_any_256_bits(bellman, oracle, log_n):
    """The coset's factors are applied first, which leaves lazy values."""
    _, dev = bellman
    x = oracle.random_fr(0xBC0000A9 + log_n, 1 << log_n)
    x[::5] = oracle.to_limbs([oracle.R - 1])[0]
    x[::7] = oracle.to_limbs([1])[0]
    got = ntt(dev, add_multiples(oracle, x, 5), log_n, log_ext=2, coset=3)
    assert np.array_equal(got, oracle.ntt(x, log_n, False, False, 2, 3))


def wide(oracle, seed, n):
    """Reduced values, and the same with up to 5 r added (no multiple of r but 0 itself)."""
    x = oracle.random_fr(seed, n)
    x[::5] = oracle.to_limbs([oracle.R - 1])[0]
    x[::7] = oracle.to_limbs([1])[0]
    return x, add_multiples(oracle, x, 5)


# every form of the inverse (blocks of 512, 2048, 4096, 8192 and 16384 elements)
@pytest.mark.parametrize("n", [2, 600, 65539, (1 << 19) + 1, (1 << 20) + 3, (1 << 21) + 5, 1 << 22, (1 << 22) + 16385])
@pytest.mark.parametrize("in_place", [False, True])
def test_batch_inverse_of_any_256_bits(bellman, oracle, n, in_place):
    B, dev = bellman
    x, y = wide(oracle, 0xBC0000B7 + n, n)
    x[3::11] = y[3::11] = 0
    if n > 65539:
        y[:n // 2] = x[:n // 2]  # whole waves of reduced elements
    d_in = dev.upload(y)
    d_out = d_in if in_place else dev.malloc(n * 32)
    B.call("ff_inverse", B.ff_inverse_configuration(dev.pool, dev.stream, d_in, d_out, n))
    dev.sync()
    got = dev.download(d_out, (n, 8))
    for p in {d_in, d_out}:
        dev.free(p)
    assert np.array_equal(got, oracle.batch_inverse(x))


# one element a thread, tiles of 1024, tiles and their products, chunks of 8
@pytest.mark.parametrize("n", [2, 255, 1000, 65539, (1 << 20) + 9, 4194299])
@pytest.mark.parametrize("every", [1, 37])
def test_prefix_products_of_any_256_bits(bellman, oracle, n, every):
    B, dev = bellman
    x, y = wide(oracle, 0xBC0000E7 + n, n)
    if every > 1:  # single elements among reduced ones
        z = x.copy()
        z[::every] = y[::every]
        y = z
    d_in, d_out = dev.upload(y), dev.malloc(n * 32)
    B.call("ff_grand_product", B.ff_grand_product_configuration(dev.pool, dev.stream, d_in, d_out, n))
    dev.sync()
    got = dev.download(d_out, (n, 8))
    dev.free(d_in)
    dev.free(d_out)
    assert np.array_equal(got, oracle.grand_product(x))


# one, two, eight and 32 elements a thread, one to three launches
@pytest.mark.parametrize("n", [2, 256, 257, 513, 2048, 2049, 65539, (1 << 17) + 1, (1 << 21) + 1, 4194299])
def test_polynomial_values_of_any_256_bits(bellman, oracle, n):
    B, dev = bellman
    x, y = wide(oracle, 0xBC0000C7 + n, n)
    point = oracle.random_fr(0xBC0000C8, 1)
    values = []
    for v in (x, y):
        d_in, d_out = dev.upload(v), dev.malloc(32)
        B.call("ff_poly_evaluate", B.ff_poly_evaluate_configuration(dev.pool, dev.stream, d_in, point.ctypes.data, d_out, n))
        dev.sync()
        values.append(dev.download(d_out, (1, 8)))
        dev.free(d_in)
        dev.free(d_out)
    assert np.array_equal(values[1], values[0])


@pytest.mark.parametrize("n", [2, 65539, (1 << 17) + 1, (1 << 20) + 7])
def test_products_with_powers_of_any_256_bits(bellman, oracle, n):
    B, dev = bellman
    x, y = wide(oracle, 0xBC0000D7 + n, n)
    base = oracle.random_fr(0xBC0000D8, 1)
    got = []
    for v in (x, y):
        d_in, d_out = dev.upload(v), dev.malloc(n * 32)
        B.call("ff_multiply_by_powers", B.ff_multiply_by_powers_configuration(dev.pool, dev.stream, d_in, base.ctypes.data, d_out, n))
        dev.sync()
        got.append(dev.download(d_out, (n, 8)))
        dev.free(d_in)
        dev.free(d_out)
    assert np.array_equal(got[1], got[0])
