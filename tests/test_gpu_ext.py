"""Extension entry points through the C ABI: fixed-base generator multiples
against the oracle's [k]G, including the comb's byte boundaries and zero."""
import ctypes

import numpy as np
import pytest

import bellman_amd as B

pytestmark = pytest.mark.gpu


def test_generator_multiples_match_oracle(bellman, oracle):
    _, dev = bellman
    R = oracle.R
    ks = [1, 2, 3, 255, 256, 257, 65535, 1 << 64, R - 1, R - 2, (1 << 253) + 12345]
    ks += [int.from_bytes(bytes((i * 37 + j * 11) & 0xFF for j in range(32)), "little") % R for i in range(53)]
    d_s = dev.upload(oracle.to_limbs(ks))
    d_p = dev.malloc(64 * len(ks))
    B.call("bc_amd_generator_multiples", ctypes.c_void_p(d_s), ctypes.c_void_p(d_p), ctypes.c_uint(len(ks)), dev.stream)
    dev.sync()
    got = dev.download(d_p, (len(ks), 16))
    for i, k in enumerate(ks):
        assert np.array_equal(got[i], oracle.mul_generator(k)), (i, k)
    dev.free(d_s)
    dev.free(d_p)


def test_generator_multiples_of_zero_are_zero_encoded(bellman, oracle):
    _, dev = bellman
    d_s = dev.upload(oracle.to_limbs([0, 0]))
    d_p = dev.malloc(128)
    B.call("bc_amd_generator_multiples", ctypes.c_void_p(d_s), ctypes.c_void_p(d_p), ctypes.c_uint(2), dev.stream)
    dev.sync()
    assert not dev.download(d_p, (2, 16)).any()
    dev.free(d_s)
    dev.free(d_p)


def fold_cases(R):
    """Discrete logs of the 254 per-bit points (0: infinity): the exceptional
    additions (equal points, opposite points, infinities) at the first, a middle
    and the last level of the fold's tree, and points everywhere."""
    single = lambda entries: [entries.get(i, 0) % R for i in range(254)]
    return {
        "infinity": single({}),
        "first bit": single({0: 5}),
        "last bit": single({253: 7}),
        "equal at the first level": single({0: 2, 1: 1}),
        "opposite at the first level": single({0: -2, 1: 1}),
        "equal at a middle level": single({8: 1 << 4, 12: 1, 200: 3}),
        "opposite at the last level": single({0: -(1 << 128), 128: 1}),
        "equal at the last level": single({3: 1 << 125, 128: 1}),
        "all one point": [1] * 254,
        "points everywhere": [pow(3, i + 1, R) for i in range(254)],
    }


def test_fold_of_exceptional_per_bit_points(bellman, oracle):
    _, dev = bellman
    R = oracle.R
    cases = fold_cases(R)
    one = oracle.to_mont([1], oracle.P)[0]
    expected, ptrs = [], []
    for logs in cases.values():
        pts = np.zeros((254, 24), dtype=np.uint32)
        for i, k in enumerate(logs):
            if k:
                pts[i, :16] = oracle.mul_generator(k)
                pts[i, 16:] = one
            else:
                pts[i, 8:16] = one
        ptrs.append(dev.upload(pts))
        total = sum(k << i for i, k in enumerate(logs)) % R
        expected.append(np.array(oracle.mul_generator(total)) if total else np.zeros(16, dtype=np.uint32))
    d_p = dev.malloc(64 * len(ptrs))
    B.call("bc_amd_msm_fold", (ctypes.c_void_p * len(ptrs))(*ptrs), ctypes.c_void_p(d_p), ctypes.c_uint(len(ptrs)), dev.stream)
    dev.sync()
    got = dev.download(d_p, (len(ptrs), 16))
    for j, name in enumerate(cases):
        assert np.array_equal(got[j], expected[j]), name
    for p in ptrs + [d_p]:
        dev.free(p)
