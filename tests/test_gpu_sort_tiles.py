"""MSM batches whose bucket sort takes the wide tiles (passes of 9 and 10 digit
bits: 7168 entries), with segments below, at and above a tile, and with every
entry in one digit; each fold equals the closed form [sum k_i s_i]G."""
import ctypes

import numpy as np
import pytest

import bellman_amd as B
from gpu_helpers import msm_batch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def based(bellman, oracle):
    _, dev = bellman
    n = 1 << 15
    logs = [pow(5, i + 1, oracle.R) for i in range(n)]
    ds, db = dev.upload(oracle.to_limbs(logs)), dev.malloc(64 * n)
    B.call("bc_amd_generator_multiples", ctypes.c_void_p(ds), ctypes.c_void_p(db), ctypes.c_uint(n), dev.stream)
    dev.sync()
    dev.free(ds)
    yield db, logs
    dev.free(db)


# one pass of 9 or 10 bits; 10 + 9, 10 + 10, 9 + 9 and 9 + 8 bits
@pytest.mark.parametrize("c", [9, 10, 17, 18, 19, 20])
def test_bucket_sort_in_wide_tiles(bellman, oracle, based, c):
    _, dev = bellman
    db, logs = based
    R = oracle.R
    jobs, scal = [], []
    for L in (2, 12, 13, 15):
        n = 1 << L
        for kind in ("random", "one value", "small"):
            k = {
                "random": [pow(7, 3 * i + L + c, R) for i in range(n)],
                "one value": [R - 12345] * n,
                "small": [i % 3 for i in range(n)],
            }[kind]
            scal.append((L, kind, k))
            jobs.append(B.msm_job(db, dev.upload(oracle.to_mont(k)), dev.malloc(254 * 96), L, c, 16))
    msm_batch(dev, jobs)
    d_p = dev.malloc(64 * len(jobs))
    B.call("bc_amd_msm_fold", (ctypes.c_void_p * len(jobs))(*[j.results for j in jobs]), ctypes.c_void_p(d_p), ctypes.c_uint(len(jobs)), dev.stream)
    dev.sync()
    got = dev.download(d_p, (len(jobs), 16))
    for j, (L, kind, k) in enumerate(scal):
        total = sum(a * b for a, b in zip(k, logs)) % R
        want = oracle.mul_generator(total) if total else np.zeros(16, dtype=np.uint32)
        assert np.array_equal(got[j], want), (L, kind)
    for job in jobs:
        dev.free(job.scalars)
        dev.free(job.results)
    dev.free(d_p)
