"""Buckets at the edges of the rules that hand them to a wave of quads (more sums
than a thread takes, up to 64), a block (up to 512) or several blocks: n equal
scalars in pieces of p entries give a bucket of n / p sums, in an ordinary place
and in the window's top digit.  Each MSM equals its closed form."""
import ctypes

import numpy as np
import pytest

import bellman_amd as B
from gpu_helpers import msm_batch

pytestmark = pytest.mark.gpu

C = 8


# sums of the bucket: 1, 4, 16, 32, 64, 128, 512, 1024 (pieces begin at the segment's start)
@pytest.mark.parametrize("log_n,piece", [(3, 8), (5, 8), (7, 8), (9, 16), (9, 8), (10, 8), (12, 8), (13, 8)])
def test_equal_scalars_fill_one_bucket(bellman, oracle, log_n, piece):
    _, dev = bellman
    n, R = 1 << log_n, oracle.R
    logs = [(11 * i * i + 5) % R for i in range(n)]
    ds, db = dev.upload(oracle.to_limbs(logs)), dev.malloc(64 * n)
    B.call("bc_amd_generator_multiples", ctypes.c_void_p(ds), ctypes.c_void_p(db), ctypes.c_uint(n), dev.stream)
    dev.sync()
    # an ordinary digit; the top digit 2^(c-1) of the first window; the last window's; one
    # entry moved out of the bucket, which shifts its run against the pieces
    values = [3, 1 << (C - 1), R - 1, (5 << C) + 3]
    scalars = [[v] * n for v in values] + [[7] + [3] * (n - 1)]
    jobs = [B.msm_job(db, dev.upload(oracle.to_mont(k)), dev.malloc(254 * 96), log_n, C, piece) for k in scalars]
    msm_batch(dev, jobs)
    for k, job in zip(scalars, jobs):
        got = dev.download(job.results, (254, 24))
        want = oracle.mul_generator(sum(a * b for a, b in zip(k, logs)) % R)
        assert np.array_equal(oracle.to_affine(oracle.msm_fold(got))[0], want), k[1]
        msm_batch(dev, [job])
        assert np.array_equal(dev.download(job.results, (254, 24)), got), k[1]
        dev.free(job.scalars)
        dev.free(job.results)
    for p in (ds, db):
        dev.free(p)
