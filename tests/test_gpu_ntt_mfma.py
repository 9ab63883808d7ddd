"""Transforms around the size where the first twelve stages move to the matrix
cores (2^18, natural order in), with inputs at the ends of the value range: the
signed digit sums there are the largest."""
import numpy as np
import pytest

from gpu_helpers import ntt, ntt_batch

pytestmark = pytest.mark.gpu


def inputs(oracle, kind, log_n):
    n = 1 << log_n
    if kind == "random":
        return oracle.random_fr(0xBC0000B1 + log_n, n)
    x = np.zeros((n, 8), dtype=np.uint32)
    top = oracle.to_limbs([oracle.R - 1])[0]  # the largest stored value
    if kind == "largest":
        x[:] = top
    elif kind == "alternating":
        x[::2] = top
    else:  # bytes 0x80 and 0x7f, where the signed digits change sign
        x[:] = 0x80808080
        x[:, 7] = 0x007F807F
        x[1::3] = 0x7F7F7F7F
        x[1::3, 7] = 0x2F7F807F
    return x


@pytest.mark.parametrize("log_n", [17, 18, 19, 21])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("kind", ["random", "largest", "alternating", "sign bytes"])
def test_natural_order_transforms(bellman, oracle, log_n, inverse, kind):
    _, dev = bellman
    x = inputs(oracle, kind, log_n)
    assert np.array_equal(ntt(dev, x, log_n, inverse=inverse), oracle.ntt(x, log_n, False, inverse))


@pytest.mark.parametrize("inverse", [False, True])
def test_cosets_in_place_and_in_a_batch(bellman, oracle, inverse):
    B, dev = bellman
    logs = [18, 10, 20, 19]
    xs = [inputs(oracle, "random", l) for l in logs]
    bufs = [dev.upload(x) for x in xs]
    ntt_batch(dev, [B.ntt_job(p, p, l, bitrev=i == 3, inverse=inverse, log_ext=2, coset=i) for i, (p, l) in enumerate(zip(bufs, logs))])
    for i, (p, x, l) in enumerate(zip(bufs, xs, logs)):
        assert np.array_equal(dev.download(p, (1 << l, 8)), oracle.ntt(x, l, i == 3, inverse, 2, i)), i
        dev.free(p)


@pytest.mark.parametrize("inverse", [False, True])
def test_third_pass(bellman, oracle, inverse):
    _, dev = bellman
    x = inputs(oracle, "random", 23)
    x[5::7] = oracle.to_limbs([oracle.R - 1])[0]
    assert np.array_equal(ntt(dev, x, 23, inverse=inverse), oracle.ntt(x, 23, False, inverse))


@pytest.mark.parametrize("log_n", [18, 19, 20, 21, 22, 24])
def test_last_pass_sizes(bellman, oracle, log_n):
    """6..10 stages are left for the last pass; the inverse's scaling and the
    coset's factors are applied there."""
    _, dev = bellman
    x = oracle.random_fr(0xBC0000E1 + log_n, 1 << log_n)
    x[7::11] = oracle.to_limbs([oracle.R - 1])[0]
    assert np.array_equal(ntt(dev, x, log_n, log_ext=1, coset=1), oracle.ntt(x, log_n, False, False, 1, 1))
    if log_n <= 22:
        assert np.array_equal(ntt(dev, x, log_n, inverse=True, log_ext=2, coset=3), oracle.ntt(x, log_n, False, True, 2, 3))
