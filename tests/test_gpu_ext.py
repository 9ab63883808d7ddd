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


def upload_per_bit(dev, oracle, rows):
    one = oracle.to_mont([1], oracle.P)[0]
    pts = np.zeros((254, 24), dtype=np.uint32)
    pts[:, 8:16] = one
    for i, xy in rows.items():
        pts[i, :16] = xy
        pts[i, 16:] = one
    return dev.upload(pts)


def fold_on_device(dev, ptrs):
    d_p = dev.malloc(64 * len(ptrs))
    B.call("bc_amd_msm_fold", (ctypes.c_void_p * len(ptrs))(*ptrs), ctypes.c_void_p(d_p), ctypes.c_uint(len(ptrs)), dev.stream)
    dev.sync()
    got = dev.download(d_p, (len(ptrs), 16))
    dev.free(d_p)
    return got


def test_fold_of_single_bits(bellman, oracle):
    """One per-bit point at every bit: 2^i, as the combination that the fold
    holds for it, times the point.  254 MSMs are several launches."""
    _, dev = bellman
    ptrs = [upload_per_bit(dev, oracle, {i: oracle.mul_generator(i + 1)}) for i in range(254)]
    got = fold_on_device(dev, ptrs)
    for i in range(254):
        assert np.array_equal(got[i], oracle.mul_generator(((i + 1) << i) % oracle.R)), i
    for p in ptrs:
        dev.free(p)


def test_fold_in_a_graph(bellman, oracle):
    """Captured, the fold takes no memory; each replay reads the results anew.
    Both counts of MSMs that the partial sums distinguish, eagerly."""
    _, dev = bellman
    hip = B.lib()  # finds the HIP functions it is linked with
    rows = [{i: oracle.mul_generator(j + i + 1) for i in range(j, 254, 11)} for j in range(7)]
    want = [oracle.mul_generator(sum((j + i + 1) << i for i in range(j, 254, 11)) % oracle.R) for j in range(7)]
    ptrs = [upload_per_bit(dev, oracle, r) for r in rows]
    for count in (1, 5, 6, 7):
        got = fold_on_device(dev, ptrs[:count])
        for j in range(count):
            assert np.array_equal(got[j], want[j]), (count, j)
    d_p = dev.malloc(64 * 7)
    graph, instance = ctypes.c_void_p(), ctypes.c_void_p()
    stream = ctypes.c_void_p(dev.stream.handle)
    assert hip.hipStreamBeginCapture(stream, ctypes.c_int(2)) == 0  # hipStreamCaptureModeRelaxed
    B.call("bc_amd_msm_fold", (ctypes.c_void_p * 7)(*ptrs), ctypes.c_void_p(d_p), ctypes.c_uint(7), dev.stream)
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(instance), graph, None, None, ctypes.c_size_t(0)) == 0
    for replay in range(3):
        assert hip.hipGraphLaunch(instance, stream) == 0
        dev.sync()
        got = dev.download(d_p, (7, 16))
        for j in range(7):
            assert np.array_equal(got[j], want[j]), (replay, j)
        fold_on_device(dev, ptrs[:2])
        B.call("bc_memset", ctypes.c_void_p(d_p), ctypes.c_int(0), ctypes.c_size_t(64 * 7))
    assert hip.hipGraphExecDestroy(instance) == 0
    assert hip.hipGraphDestroy(graph) == 0
    for p in ptrs + [d_p]:
        dev.free(p)


def test_fold_of_points_off_the_curve(bellman, oracle):
    """Points of y^2 = x^3 + 17, where the curve's endomorphism does not act:
    the fold is still the integer combination, by the same affine formulas."""
    _, dev = bellman
    p = oracle.P

    def add(a, b):
        if a is None or b is None:
            return a or b
        if a[0] == b[0]:
            if (a[1] + b[1]) % p == 0:
                return None
            m = 3 * a[0] * a[0] * pow(2 * a[1], -1, p)
        else:
            m = (b[1] - a[1]) * pow(b[0] - a[0], -1, p)
        x = (m * m - a[0] - b[0]) % p
        return x, (m * (a[0] - x) - a[1]) % p

    base = (p - 2, 3)  # 9 = -8 + 17
    points, q = [], base
    for _ in range(254):
        points.append(q)
        q = add(q, base)
    total = None
    for q in reversed(points):
        total = add(add(total, total), q)
    limbs = lambda q: np.concatenate([oracle.to_mont([q[0]], p)[0], oracle.to_mont([q[1]], p)[0]])
    on = {i: oracle.mul_generator(i + 1) for i in range(254)}
    ptrs = [upload_per_bit(dev, oracle, {i: limbs(q) for i, q in enumerate(points)}), upload_per_bit(dev, oracle, on)]
    got = fold_on_device(dev, ptrs)
    assert np.array_equal(got[0], limbs(total))
    assert np.array_equal(got[1], oracle.mul_generator(sum((i + 1) << i for i in range(254)) % oracle.R))
    for ptr in ptrs:
        dev.free(ptr)
