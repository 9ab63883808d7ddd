"""Field inversion: the divsteps routine (csrc/inverse.cuh) on the host against
Python integers, and ff_inverse on the device at the edges of its blocks."""
import ctypes
import os
import random
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HARNESS = os.path.join(ROOT, "tests", "hostinv", "harness.hip")
HIPCC = "/opt/rocm/bin/hipcc"
P = 21888242871839275222246405745257275088696311157297823662689037894645226208583
R = 21888242871839275222246405745257275088548364400416034343698204186575808495617


@pytest.mark.parametrize("base_field,m", [(1, P), (0, R)])
def test_divsteps_inverse_on_the_host(tmp_path, base_field, m):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path / "libhostinv.so")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-fPIC", "-shared", "--offload-arch=gfx950", HARNESS, "-o", out], check=True, capture_output=True)
    lib = ctypes.CDLL(out)
    rng = random.Random(0xBC2902)
    values = [0, 1, 2, m - 1, m - 2, m, m + 1, 2 * m - 1, (m - 1) // 2] + [1 << i for i in range(254)] + [m - (1 << i) for i in range(253)]
    values += [rng.randrange(2 * m) for _ in range(2000)]
    for x in values:
        a = np.array([(x >> (32 * i)) & 0xFFFFFFFF for i in range(8)], dtype=np.uint32)
        r = np.zeros(8, dtype=np.uint32)
        lib.hostinv(base_field, a.ctypes.data_as(ctypes.c_void_p), r.ctypes.data_as(ctypes.c_void_p))
        expected = pow(x, -1, m) * (1 << 512) % m if x % m else 0
        assert sum(int(w) << (32 * i) for i, w in enumerate(r)) == expected, x


# blocks of 512 elements up to 2^19, 2048 up to 2^20, 4096 up to 2^21, 8192 above
@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 256, 257, 511, 512, 513, 65539, 1 << 19, (1 << 19) + 1, 1 << 20, (1 << 20) + 4097, (1 << 21) + 8191])
@pytest.mark.parametrize("in_place", [False, True])
def test_batch_inverse_at_block_edges(bellman, oracle, n, in_place):
    B, dev = bellman
    x = oracle.random_fr(n + 7, n)
    x[n - 1] = 0
    x[n // 2:n // 2 + 600:3] = 0
    if n > 4096:
        x[1024:3072] = 0  # whole blocks of zeros
    x[0] = oracle.to_mont([R - 1])[0]
    dx = dev.upload(x)
    dy = dx if in_place else dev.malloc(n * 32)
    B.call("ff_inverse", B.ff_inverse_configuration(dev.pool, dev.stream, dx, dy, n))
    dev.sync()
    assert np.array_equal(dev.download(dy, (n, 8)), oracle.batch_inverse(x))
    dev.free(dx)
    if not in_place:
        dev.free(dy)
