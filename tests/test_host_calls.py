"""What the library asks of the HIP runtime, and in which order, read on the CPU:
libbellman.so is loaded over a runtime that runs nothing and lists the calls it
gets (tests/hostrt/fake_hip.cpp).  Each test is a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "era-bellman-cuda_amd")

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(%r, mode=ctypes.RTLD_GLOBAL)  # before libbellman.so, whose runtime calls it takes
fake.fake_log.restype = ctypes.c_char_p
import bellman_amd as B
DEVICE = 32 << 40  # an address in device 0's memory
PEER = 33 << 40    # and in device 1's

def calls():
    lines = fake.fake_log().decode().splitlines()
    fake.fake_clear()
    return [l.split() for l in lines]

def stream_of(call):
    return call[-1]

def set_up():
    B.call("ff_set_up", ctypes.c_uint(25), ctypes.c_uint(14))
    B.call("ntt_set_up")
    s = B.bc_stream()
    B.call("bc_stream_create", ctypes.byref(s), ctypes.c_bool(False))
    fake.fake_clear()
    return s
"""


@pytest.fixture(scope="session")
def run(tmp_path_factory):
    """Runs a snippet in a process whose HIP runtime is the listing one."""
    import bellman_amd as B

    if not os.path.exists(B.LIB_PATH):
        pytest.skip("libbellman.so not built")
    fake = str(tmp_path_factory.mktemp("hostrt") / "libfakehip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-attributes",
                    os.path.join(ROOT, "tests", "hostrt", "fake_hip.cpp"), "-o", fake], check=True, capture_output=True)

    def go(body):
        p = subprocess.run([sys.executable, "-c", PRELUDE % fake + body], capture_output=True, text=True, env=dict(os.environ, PYTHONPATH=os.pathsep.join((PKG, ROOT))), timeout=120)
        assert p.returncode == 0, p.stdout + p.stderr

    return go


@pytest.mark.parametrize("log_n", [20, 22])
def test_staging_memory_is_released_after_the_copies(run, log_n):
    """An MSM over host inputs that fails with a chunk's copy still running on
    the copy stream: the call's stream waits for that stream before it gives the
    staging memory back."""
    run("""
s = set_up()
cfg = B.msm_configuration()
scalars = ctypes.create_string_buffer(32)  # not read: copies are only listed
cfg.stream, cfg.bases, cfg.scalars, cfg.results, cfg.log_scalars_count = s, DEVICE, ctypes.addressof(scalars), DEVICE, %d
cfg.h2d_copy_finished_callback = B.bc_host_fn(lambda data: None)
fake.fake_fail(b"host_func")  # enqueued after the last copy, before the call's stream waits for it
assert B.lib().msm_execute_async(cfg) != 0
log = calls()
mine = "s=%%x" %% s.handle
last = max(i for i, c in enumerate(log) if c[0] == "memcpy")
side = stream_of(log[last])
assert side != mine
freed = min(i for i, c in enumerate(log) if c[0] == "free_async" and i > last)
events = [c[1] for c in log[last:freed] if c[0] == "record" and c[2] == side]
waits = [c[1] for c in log[last:freed] if c[0] == "wait" and c[2] == mine]
assert set(events) & set(waits), log[last:]
""" % log_n)


@pytest.mark.parametrize("log_n", [4, 18, 20])
def test_a_finished_msm_does_not_wait_for_the_callback(run, log_n):
    """Where the call succeeds, its stream waits for the copies (events recorded
    before the callback), not for the callback after them."""
    run("""
s = set_up()
cfg = B.msm_configuration()
scalars = ctypes.create_string_buffer(32)
cfg.stream, cfg.bases, cfg.scalars, cfg.results, cfg.log_scalars_count = s, DEVICE, ctypes.addressof(scalars), DEVICE, %d
cfg.h2d_copy_finished_callback = B.bc_host_fn(lambda data: None)
B.call("msm_execute_async", cfg)
log = calls()
mine = "s=%%x" %% s.handle
at = next(i for i, c in enumerate(log) if c[0] == "host_func")
assert log[at][1] != mine
after = [c[1] for c in log[at:] if c[0] == "record" and c[2] == log[at][1]]
assert not [c for c in log if c[0] == "wait" and c[2] == mine and c[1] in after]
""" % log_n)


@pytest.mark.parametrize("count", [0, 100, 65539, 1 << 22])
@pytest.mark.parametrize("where", ["own", "peer", "host"])
def test_a_polynomial_value_for_another_gpu_is_copied(run, count, where):
    """Kernels write a result in the memory of the stream's GPU; one in the host's
    or another GPU's memory, which no kernel here may reach, is copied."""
    run("""
s = set_up()
host = ctypes.create_string_buffer(32)
result = {"own": DEVICE + 4096, "peer": PEER, "host": ctypes.addressof(host)}[%r]
point = (ctypes.c_uint * 8)(3)
B.call("ff_poly_evaluate", B.ff_poly_evaluate_configuration(B.bc_mem_pool(), s, DEVICE, ctypes.addressof(point), result, %d))
copies = [c for c in calls() if c[0] == "memcpy"]
assert [int(c[1], 16) for c in copies] == ([] if result == DEVICE + 4096 else [result])
assert all(c[3] == "32" and stream_of(c) == "s=%%x" %% s.handle for c in copies)
""" % (where, count))


def test_at_most_one_element_needs_no_scalar(run):
    """The only power of the point or base is then the 0th."""
    run("""
s = set_up()
pool = B.bc_mem_pool()
for n in (0, 1):
    B.call("ff_poly_evaluate", B.ff_poly_evaluate_configuration(pool, s, DEVICE, None, DEVICE + 4096, n))
    assert [c[0] for c in calls()] == ["launch"]
B.call("ff_multiply_by_powers", B.ff_multiply_by_powers_configuration(pool, s, DEVICE, None, DEVICE + 4096, 1))
assert [c[0] for c in calls()] == ["launch"]
""")


@pytest.mark.gpu
def test_one_element_with_and_without_a_scalar(bellman, oracle):
    import ctypes

    import numpy as np

    B, dev = bellman
    x = oracle.random_fr(0xBC0000F1, 1)
    dx, dy = dev.upload(x), dev.malloc(32)
    point = oracle.random_fr(0xBC0000F2, 1)
    for p in (None, point.ctypes.data):
        for name in ("ff_poly_evaluate", "ff_multiply_by_powers"):
            B.call("bc_memset", B.ptr(dy), ctypes.c_int(0x5A), ctypes.c_size_t(32))
            if name == "ff_poly_evaluate":
                B.call(name, B.ff_poly_evaluate_configuration(dev.pool, dev.stream, dx, p, dy, 1))
            else:
                B.call(name, B.ff_multiply_by_powers_configuration(dev.pool, dev.stream, dx, p, dy, 1))
            dev.sync()
            assert np.array_equal(dev.download(dy, (1, 8)), x), name
    for p in (dx, dy):
        dev.free(p)


NTT = """
def transform(log_n, inverse, bitrev=False, log_ext=0):
    cfg = B.ntt_configuration()
    cfg.stream, cfg.inputs, cfg.outputs, cfg.log_values_count, cfg.inverse, cfg.bit_reversed_inputs = s, DEVICE, DEVICE, log_n, inverse, bitrev
    cfg.log_extension_degree = log_ext
    B.call("ntt_execute_async", cfg)
    return calls()

def kernels(log):
    return [c[1] for c in log if c[0] == "launch"]

def waits_or_allocates(log):
    return [c for c in log if c[0] in ("malloc", "synchronize", "device")]
"""


def test_transforms_neither_allocate_nor_wait(run):
    """Up to the size that the tables were made for, from the first transform on,
    with and without the field's power tables."""
    run(NTT + """
s = set_up()
for tear_down in (False, True):
    if tear_down:
        B.call("ff_tear_down")
        calls()
    for log_n in (12, 17, 18, 19, 20):
        for inverse in (False, True):
            log = transform(log_n, inverse)
            assert [c[0] for c in log] == ["launch"] * len(log), log
            assert any("ntt_mfma_last" in k for k in kernels(log)) == (log_n >= 18)
""")


def test_one_growth_makes_every_table(run):
    run(NTT + """
s = set_up()
grown = transform(24, False)
assert waits_or_allocates(grown)
for log_n in (18, 21, 22, 23, 24):
    for inverse in (False, True):
        log = transform(log_n, inverse)
        assert not waits_or_allocates(log), log
        assert any("ntt_mfma_last" in k for k in kernels(log)) == (log_n != 23)
B.call("ntt_tear_down")
freed = [c for c in calls() if c[0] == "free"]
# twiddles of both sizes, powers of 1/2, matrices, row factors of the third pass and of the last pass of six sizes
assert len(freed) == 2 + 2 + 1 + 1 + 1 + 12 and len(set(c[1] for c in freed)) == len(freed)
""")


def test_a_nearly_full_gpu_keeps_its_memory(run):
    """Without room to spare the last stages are VALU passes, and no call tries again."""
    run(NTT + """
fake.fake_memory(ctypes.c_size_t(30 << 30), ctypes.c_size_t(256 << 30))
s = set_up()
transform(24, True)
for log_n in (18, 20, 22, 24):
    for inverse in (False, True):
        log = transform(log_n, inverse)
        assert not waits_or_allocates(log), log
        names = kernels(log)
        assert not any("ntt_mfma_last" in k for k in names) and any("ntt_pass_kernel" in k for k in names) and "ntt_mfma" in names[0], names
""")


def test_grand_product_where_the_pool_is_small(run):
    """4194299 elements: 16 MiB of chunk products, or 132 KiB of tile products where
    the pool has no more."""
    run("""
s = set_up()
cfg = B.ff_grand_product_configuration(B.bc_mem_pool(), s, DEVICE, DEVICE, 4194299)
B.call("ff_grand_product", cfg)
assert any("chunk" in c[1] for c in calls() if c[0] == "launch")
fake.fake_largest(ctypes.c_size_t(1 << 20))
B.call("ff_grand_product", cfg)
log = calls()
names = [c[1] for c in log if c[0] == "launch"]
assert len(names) == 5 and not any("chunk" in k or "apply" in k for k in names), names
assert sorted(c[1] for c in log if c[0] == "malloc_async" and c[1] != "refused") == sorted(c[1] for c in log if c[0] == "free_async")
fake.fake_largest(ctypes.c_size_t(1 << 10))
assert B.lib().ff_grand_product(cfg) == B.bc_error_memory_allocation
""")


@pytest.mark.gpu
def test_grand_product_from_a_pool_of_four_mebibytes(bellman, oracle):
    import ctypes

    import numpy as np

    B, dev = bellman

    class pool_properties(ctypes.Structure):  # hipMemPoolProps
        _fields_ = [("type", ctypes.c_int), ("handles", ctypes.c_int), ("location", ctypes.c_int), ("device", ctypes.c_int),
                    ("attributes", ctypes.c_void_p), ("most", ctypes.c_size_t), ("reserved", ctypes.c_ubyte * 56)]

    pool = B.bc_mem_pool()
    assert B.lib().hipMemPoolCreate(ctypes.byref(pool), ctypes.byref(pool_properties(type=1, location=1, device=0, most=4 << 20))) == 0
    n = 4194299
    x = oracle.random_fr(0xBC0000F9, n)
    dx, dy = dev.upload(x), dev.malloc(n * 32)
    p = ctypes.c_void_p()
    assert B.lib().bc_malloc_from_pool_async(ctypes.byref(p), ctypes.c_size_t(16 << 20), pool, dev.stream) == B.bc_error_memory_allocation
    B.call("ff_grand_product", B.ff_grand_product_configuration(pool, dev.stream, dx, dy, n))
    dev.sync()
    assert np.array_equal(dev.download(dy, (n, 8)), oracle.grand_product(x))
    B.call("bc_mem_pool_destroy", pool)
    dev.free(dx)
    dev.free(dy)


def test_plain_msm_memory_is_its_footprint(run):
    """The one block that a plain MSM takes is the footprint of its window width
    with some chunk of sorted entries, the chunk grows with the size, and the largest
    call of the fixed array is the last whose footprint fits it."""
    run("""
from oracle import oracle as O
s = set_up()
def footprint(log_n, piece):
    job, out = B.bc_amd_job(), ctypes.c_size_t()
    job.kind, job.msm = B.BC_AMD_JOB_MSM, B.msm_job(DEVICE, DEVICE, DEVICE, log_n, O.msm_window_bits(log_n), piece)
    B.call("bc_amd_job_footprint", ctypes.byref(job), ctypes.byref(out))
    return out.value
taken, pieces = [], []
for log_n in range(27):
    cfg = B.msm_configuration()
    cfg.stream, cfg.bases, cfg.scalars, cfg.results, cfg.log_scalars_count = s, DEVICE, DEVICE, DEVICE, log_n
    B.call("msm_execute_async", cfg)
    blocks = [int(c[2]) for c in calls() if c[0] == "malloc_async"]
    fitting = [p for p in (4, 8, 16, 32, 64, 128) if footprint(log_n, p) == blocks[0]]
    assert len(blocks) == 1 and fitting, (log_n, blocks)
    taken.append(blocks[0])
    pieces.append(max(fitting))
assert all(a <= b for a, b in zip(pieces[10:], pieces[11:])) and pieces[26] == 128, pieces
for log_n in (16, 17, 18):
    cfg.log_scalars_count = log_n
    fits = taken[log_n] <= 192 << 20
    assert fits == (log_n <= 17)
    assert (B.lib().bc_amd_msm_execute_no_alloc(cfg) == B.bc_success) == fits
    assert not [c for c in calls() if c[0].startswith("malloc")]
""")


def test_four_chunks_of_host_inputs_reuse_two_slots(run):
    """At 2^22 points the copy of chunk k + 2 waits for the kernels of chunk k."""
    run("""
s = set_up()
scalars = ctypes.create_string_buffer(32)
cfg = B.msm_configuration()
cfg.stream, cfg.bases, cfg.scalars, cfg.results, cfg.log_scalars_count = s, DEVICE, ctypes.addressof(scalars), DEVICE, 22
B.call("msm_execute_async", cfg)
log = calls()
mine = "s=%x" % s.handle
copies = [i for i, c in enumerate(log) if c[0] == "memcpy"]
assert [int(log[i][3]) for i in copies] == [32 << 20] * 4
assert log[copies[0]][1] == log[copies[2]][1] != log[copies[1]][1] == log[copies[3]][1]
side = stream_of(log[copies[0]])
accumulated = [i for i, c in enumerate(log) if c[0] == "launch" and "bucket_gather" in c[1]]
assert len(accumulated) == 4 and all(stream_of(log[i]) == mine for i in accumulated)
for k in (2, 3):
    waits = [c[1] for c in log[copies[k - 1]:copies[k]] if c[0] == "wait" and c[2] == side]
    freed = [c[1] for c in log[accumulated[k - 2]:copies[k]] if c[0] == "record" and c[2] == mine]
    assert set(waits) & set(freed), (k, log[copies[k - 1]:copies[k]])
for k in range(4):  # and a chunk's kernels wait for its copy
    loaded = [c[1] for c in log[copies[k]:] if c[0] == "record" and c[2] == side][0]
    digits = [i for i, c in enumerate(log) if c[0] == "launch" and "digits" in c[1]][k]
    assert any(c[0] == "wait" and c[1] == loaded and c[2] == mine for c in log[copies[k]:digits])
""")
