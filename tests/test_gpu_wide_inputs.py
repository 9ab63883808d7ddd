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
