"""Workloads of a PLONK prover over BN254, as its program drives libbellman.

A case is a dict of plain values.  `prepare` makes what the program holds before
the call (inputs on the device, the memory pool, a batch's plan), `run` makes one
pass through the C ABI on torch's current stream, `work` counts what the pass
cannot do without and `exact` recomputes the outputs with Python integers.

Kinds:
  ntt               one Fr transform (ntt_execute_async): either input order,
                    either direction, optionally on a coset
  lde               a column's way from its values on the domain to its values on
                    every coset of the extended domain: inverse transform,
                    bit reversal, one coset transform per coset
  msm               one polynomial commitment (msm_execute_async, then the fold of
                    its 254 per-bit points into the committed point); the scalars
                    are device memory or a pinned host buffer
  pn                the permutation polynomials of a circuit
  copy_permutation  the grand product z(X) of the permutation argument, from the
                    element-wise ops, the batch inverse and the prefix product
  opening           evaluations of several polynomials at one point, their random
                    linear combination, and its variable scaled by that point
  batch             many uneven MSMs and NTTs as one plan replay, every MSM folded

Field elements are int32 tensors of shape (n, 8): little-endian limbs, Montgomery
form with R = 2^256.  The per-bit points of an MSM are Jacobian, so their
coordinates are not unique; the folded point is affine and canonical, and it is
what a commitment is.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "era-bellman-cuda_amd"))
import bellman_amd as B  # noqa: E402

P = 21888242871839275222246405745257275088696311157297823662689037894645226208583
R = 21888242871839275222246405745257275088548364400416034343698204186575808495617
MONT = 1 << 256
TOP_LIMB = 0x30644E72  # top limb of r: limbs with a smaller top one are canonical
GENERATOR = 7
ROOT_2_28 = pow(GENERATOR, (R - 1) >> 28, R)
PRODUCT_OPS = 2 * 136  # 32-bit multiply-adds of one field product, two operations each


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest transform a prover issues: latency and launches
        {"name": "ntt_2e12", "kind": "ntt", "log_n": 12, "bit_reversed": False, "inverse": False, "log_ext": 0, "coset": 0},
        # back from bit-reversed evaluations to coefficients, a mid-sized circuit
        {"name": "intt_bitrev_2e17", "kind": "ntt", "log_n": 17, "bit_reversed": True, "inverse": True, "log_ext": 0, "coset": 0},
        # the headline transform
        {"name": "ntt_2e24", "kind": "ntt", "log_n": 24, "bit_reversed": False, "inverse": False, "log_ext": 0, "coset": 0},
        # one witness column of a 2^20-row circuit, extended four times
        {"name": "lde4_2e20", "kind": "lde", "log_n": 20, "log_ext": 2},
        # commitment of a small circuit: launches, short reductions, the fold
        {"name": "msm_2e12", "kind": "msm", "log_n": 12, "host_scalars": False},
        # commitment of a column that still lies in pinned host memory
        {"name": "msm_host_2e18", "kind": "msm", "log_n": 18, "host_scalars": True},
        # commitment of a 2^20-row column
        {"name": "msm_2e20", "kind": "msm", "log_n": 20, "host_scalars": False},
        # the headline commitment
        {"name": "msm_2e24", "kind": "msm", "log_n": 24, "host_scalars": False},
        # set-up of a four-column circuit with 2^20 rows
        {"name": "pn_4x2e20", "kind": "pn", "columns": 4, "log_rows": 20},
        # permutation argument of a large circuit, the blinded rows left out
        {"name": "copy_permutation_4194299", "kind": "copy_permutation", "columns": 4, "count": 4194299},
        # openings of a small circuit's polynomials, degree raised by the blinding
        {"name": "opening_8x65539", "kind": "opening", "polys": 8, "count": 65539},
        # many small proofs side by side
        {"name": "batch_24msm_12ntt", "kind": "batch", "msms": 24, "msm_log_min": 12, "msm_log_max": 17, "ntts": 12, "ntt_log_min": 10, "ntt_log_max": 20},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["ntt", "ntt", "lde", "msm", "msm", "pn", "copy_permutation", "copy_permutation", "opening", "opening", "batch"])
    if kind == "ntt":
        log_n = rng.randint(8, 24)
        log_ext = rng.choice([0, 0, 1, 2, 3])
        return {"kind": kind, "log_n": log_n, "bit_reversed": rng.random() < 0.5, "inverse": rng.random() < 0.5, "log_ext": log_ext,
                "coset": rng.randrange(1 << log_ext)}
    if kind == "lde":
        return {"kind": kind, "log_n": rng.randint(10, 21), "log_ext": rng.randint(1, 3)}
    if kind == "msm":
        return {"kind": kind, "log_n": rng.randint(8, 22), "host_scalars": rng.random() < 0.25}
    if kind == "pn":
        return {"kind": kind, "columns": rng.choice([3, 4]), "log_rows": rng.randint(10, 22)}
    if kind == "copy_permutation":
        return {"kind": kind, "columns": rng.choice([3, 4]), "count": _log_uniform(rng, 300, 1 << 23)}
    if kind == "opening":
        return {"kind": kind, "polys": rng.randint(2, 12), "count": _log_uniform(rng, 300, 1 << 22)}
    low = rng.randint(10, 13)
    return {"kind": kind, "msms": rng.randint(4, 32), "msm_log_min": low, "msm_log_max": low + rng.randint(1, 4), "ntts": rng.randint(2, 24),
            "ntt_log_min": rng.randint(8, 12), "ntt_log_max": rng.randint(13, 20)}


def _spread(low, high, count):
    """`count` log sizes from low to high, evenly."""
    return [low + (i * (high - low) + (count - 1) // 2) // max(count - 1, 1) for i in range(count)]


# ---------------------------------------------------------------- the program's side of the C ABI
_pool = None


def _library():
    """Tables and the memory pool, set up once as a program does at start."""
    global _pool
    if _pool is None:
        torch.cuda.init()
        torch.empty(1, device="cuda")
        B.call("bc_set_device", ctypes.c_int(torch.cuda.current_device()))
        B.call("ff_set_up", ctypes.c_uint(25), ctypes.c_uint(14))
        for name in ("ntt_set_up", "pn_set_up", "msm_set_up"):
            B.call(name)
        pool = B.bc_mem_pool()
        B.call("bc_mem_pool_create", ctypes.byref(pool), ctypes.c_int(torch.cuda.current_device()))
        _pool = pool
    return _pool


def _stream():
    return B.bc_stream(torch.cuda.current_stream().cuda_stream)


def _vp(tensor):
    return ctypes.c_void_p(tensor.data_ptr())


def _u(v):
    return ctypes.c_uint(v)


def _elements(*shape):
    return torch.empty(shape + (8,), dtype=torch.int32, device="cuda")


def _limbs(values):
    data = b"".join(v.to_bytes(32, "little") for v in values)
    return np.frombuffer(data, dtype=np.uint32).reshape(-1, 8).copy()


def _scalar(value):
    """A field element in host memory (Montgomery form)."""
    return _limbs([value * MONT % R])


# ---------------------------------------------------------------- inputs, from the seed alone
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _random_fr(g, n):
    """n canonical values below r, uniform over all limbs."""
    x = torch.randint(-(1 << 31), 1 << 31, (n, 8), dtype=torch.int32, device="cuda", generator=g)
    x[:, 7] = torch.randint(0, TOP_LIMB, (n,), dtype=torch.int32, device="cuda", generator=g)
    return x


def _witness_scalars(g, n):
    """Values as a witness column has them: 70 % uniform, 20 % below 2^64, 10 % zero or one."""
    x = _random_fr(g, n)
    sort = torch.rand(n, device="cuda", generator=g)
    x[:, 2:] = torch.where((sort >= 0.7).unsqueeze(1), torch.zeros_like(x[:, 2:]), x[:, 2:])
    bit = sort >= 0.9
    x[:, 1] = torch.where(bit, torch.zeros_like(x[:, 1]), x[:, 1])
    x[:, 0] = torch.where(bit, x[:, 0] & 1, x[:, 0])
    return x


def _to_montgomery(x):
    out = torch.empty_like(x)
    r2 = _limbs([MONT * MONT % R])
    B.call("ff_ax", B.ptr(r2), _vp(x), _vp(out), _u(x.shape[0]), _stream())
    return out


def _bases(discrete_logs):
    """Affine points [s] G."""
    n = discrete_logs.shape[0]
    points = torch.empty((n, 16), dtype=torch.int32, device="cuda")
    B.call("bc_amd_generator_multiples", _vp(discrete_logs), _vp(points), _u(n), _stream())
    return points


def _cycles(g, cells):
    """Variable indexes in random cycles of 1..64 cells."""
    order = torch.randperm(cells, device="cuda", generator=g)
    lengths = torch.randint(1, 65, (cells // 16 + 64,), device="cuda", generator=g)
    ends = torch.cumsum(lengths, 0)
    variable = torch.searchsorted(ends, torch.arange(cells, device="cuda"), right=True).to(torch.int32)
    indexes = torch.empty(cells, dtype=torch.int32, device="cuda")
    indexes[order] = variable
    return indexes


def _challenges(seed, count):
    """Field elements as a transcript gives them, in host memory."""
    rng = np.random.default_rng(seed)
    return [int.from_bytes(rng.bytes(32), "little") % R for _ in range(count)]


def _inputs(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind in ("ntt", "lde"):
        return {"values": _random_fr(g, 1 << case["log_n"])}
    if kind == "msm":
        n = 1 << case["log_n"]
        return {"logs": _random_fr(g, n), "scalars": _witness_scalars(g, n)}
    if kind == "pn":
        return {"indexes": _cycles(g, case["columns"] << case["log_rows"]), "factors": _random_fr(g, case["columns"])}
    if kind == "copy_permutation":
        k, n = case["columns"], case["count"]
        return {"witness": [_random_fr(g, n) for _ in range(k)], "sigma": [_random_fr(g, n) for _ in range(k)], "challenges": _challenges(seed, k + 2)}
    if kind == "opening":
        return {"polys": [_random_fr(g, case["count"]) for _ in range(case["polys"])], "challenges": _challenges(seed, 2)}
    msm_logs = _spread(case["msm_log_min"], case["msm_log_max"], case["msms"])
    ntt_logs = _spread(case["ntt_log_min"], case["ntt_log_max"], case["ntts"])
    return {"logs": _random_fr(g, 1 << max(msm_logs)), "scalars": [_witness_scalars(g, 1 << l) for l in msm_logs],
            "values": [_random_fr(g, 1 << l) for l in ntt_logs], "msm_logs": msm_logs, "ntt_logs": ntt_logs}


def _ntt_configuration(source, target, log_n, bit_reversed=False, inverse=False, log_ext=0, coset=0):
    cfg = B.ntt_configuration()
    cfg.mem_pool = _pool
    cfg.inputs = source.data_ptr()
    cfg.outputs = target.data_ptr()
    cfg.log_values_count = log_n
    cfg.bit_reversed_inputs = bit_reversed
    cfg.inverse = inverse
    cfg.log_extension_degree = log_ext
    cfg.coset_index = coset
    return cfg


class _Plan:
    """A captured batch, released with its owner."""

    def __init__(self, msm_jobs, ntt_jobs):
        self.handle = B.bc_amd_plan()
        B.call("bc_amd_plan_create", ctypes.byref(self.handle), B.array_of(B.bc_amd_msm_job, msm_jobs), _u(len(msm_jobs)),
               B.array_of(B.bc_amd_ntt_job, ntt_jobs), _u(len(ntt_jobs)))

    def __del__(self):
        if self.handle.handle:
            B.lib().bc_amd_plan_destroy(self.handle)


def prepare(case, seed):
    _library()
    kind = case["kind"]
    state = dict(case)
    x = _inputs(case, seed)
    if kind == "ntt":
        state["values"] = x["values"]
        state["out"] = torch.empty_like(x["values"])
        state["cfg"] = _ntt_configuration(state["values"], state["out"], case["log_n"], case["bit_reversed"], case["inverse"], case["log_ext"], case["coset"])
    elif kind == "lde":
        n = 1 << case["log_n"]
        state["values"] = x["values"]
        state["reversed"], state["coefficients"] = _elements(n), _elements(n)
        state["out"] = _elements(1 << case["log_ext"], n)
        state["inverse_cfg"] = _ntt_configuration(state["values"], state["reversed"], case["log_n"], inverse=True)
        state["coset_cfgs"] = [_ntt_configuration(state["coefficients"], state["out"][c], case["log_n"], log_ext=case["log_ext"], coset=c)
                               for c in range(1 << case["log_ext"])]
    elif kind == "msm":
        scalars = _to_montgomery(x["scalars"])
        if case["host_scalars"]:
            host = torch.empty(scalars.shape, dtype=torch.int32, pin_memory=True)
            host.copy_(scalars)
            scalars = host
        state["bases"], state["scalars"] = _bases(x["logs"]), scalars
        state["bits"] = torch.empty((254, 24), dtype=torch.int32, device="cuda")
        state["point"] = torch.empty((1, 16), dtype=torch.int32, device="cuda")
        state["results"] = (ctypes.c_void_p * 1)(state["bits"].data_ptr())
        cfg = B.msm_configuration()
        cfg.mem_pool = _pool
        cfg.bases, cfg.scalars, cfg.results = state["bases"].data_ptr(), scalars.data_ptr(), state["bits"].data_ptr()
        cfg.log_scalars_count = case["log_n"]
        state["cfg"] = cfg
    elif kind == "pn":
        state.update(x)
        state["out"] = _elements(case["columns"], 1 << case["log_rows"])
        state["cfg"] = B.generate_permutation_polynomials_configuration(_pool, B.bc_stream(), x["indexes"].data_ptr(), x["factors"].data_ptr(),
                                                                        state["out"].data_ptr(), case["columns"], case["log_rows"])
    elif kind == "copy_permutation":
        state.update(x)
        n = case["count"]
        state["log_degree"] = max(n - 1, 1).bit_length()
        for name in ("domain", "term", "numerator", "denominator", "inverse", "ratio", "z"):
            state[name] = _elements(n)
        beta, gamma = x["challenges"][:2]
        state["beta"], state["gamma"] = _scalar(beta), _scalar(gamma)
        # beta times the coset factor of each column (the first column's is 1)
        state["beta_k"] = [_scalar(beta)] + [_scalar(beta * k % R) for k in x["challenges"][2:2 + case["columns"] - 1]]
    elif kind == "opening":
        state.update(x)
        z, v = x["challenges"]
        state["z"] = _scalar(z)
        state["v_powers"] = [_scalar(pow(v, i, R)) for i in range(case["polys"])]
        state["evaluations"] = _elements(case["polys"])
        state["combined"], state["scaled"] = _elements(case["count"]), _elements(case["count"])
    else:
        bases = _bases(x["logs"])
        scalars = [_to_montgomery(s) for s in x["scalars"]]
        bits = torch.empty((case["msms"], 254, 24), dtype=torch.int32, device="cuda")
        outs = [torch.empty_like(v) for v in x["values"]]
        state.update(bases=bases, scalars=scalars, bits=bits, values=x["values"], outs=outs)
        state["points"] = torch.empty((case["msms"], 16), dtype=torch.int32, device="cuda")
        state["results"] = (ctypes.c_void_p * case["msms"])(*[bits[i].data_ptr() for i in range(case["msms"])])
        state["plan"] = _Plan([B.msm_job(bases.data_ptr(), s.data_ptr(), bits[i].data_ptr(), l) for i, (s, l) in enumerate(zip(scalars, x["msm_logs"]))],
                              [B.ntt_job(v.data_ptr(), o.data_ptr(), l) for v, o, l in zip(x["values"], outs, x["ntt_logs"])])
    return state


# ---------------------------------------------------------------- one pass
def run(state):
    kind, stream = state["kind"], _stream()
    if kind == "ntt":
        state["cfg"].stream = stream
        B.call("ntt_execute_async", state["cfg"])
        return state["out"]
    if kind == "lde":
        state["inverse_cfg"].stream = stream
        B.call("ntt_execute_async", state["inverse_cfg"])
        B.call("ff_bit_reverse", _vp(state["reversed"]), _vp(state["coefficients"]), _u(state["log_n"]), stream)
        for cfg in state["coset_cfgs"]:
            cfg.stream = stream
            B.call("ntt_execute_async", cfg)
        return {"coefficients": state["coefficients"], "cosets": state["out"]}
    if kind == "msm":
        state["cfg"].stream = stream
        B.call("msm_execute_async", state["cfg"])
        B.call("bc_amd_msm_fold", state["results"], _vp(state["point"]), _u(1), stream)
        return state["point"]
    if kind == "pn":
        state["cfg"].stream = stream
        B.call("pn_generate_permutation_polynomials", state["cfg"])
        return state["out"]
    if kind == "copy_permutation":
        return _run_copy_permutation(state, stream)
    if kind == "opening":
        return _run_opening(state, stream)
    B.call("bc_amd_plan_launch", state["plan"].handle, stream)
    B.call("bc_amd_msm_fold", state["results"], _vp(state["points"]), _u(state["msms"]), stream)
    return {"points": state["points"], "transforms": state["outs"]}


def _run_copy_permutation(s, stream):
    """z[i] = prod over j <= i, columns c of (w + beta k_c omega^j + gamma) / (w + beta sigma_c + gamma)."""
    n = _u(s["count"])
    domain, term, num, den, inv = (_vp(s[name]) for name in ("domain", "term", "numerator", "denominator", "inverse"))
    B.call("ff_get_powers_of_w", domain, _u(s["log_degree"]), _u(0), n, ctypes.c_bool(False), ctypes.c_bool(False), stream)
    for c in range(s["columns"]):
        for side, factor, values in ((num, s["beta_k"][c], domain), (den, s["beta"], _vp(s["sigma"][c]))):
            into = side if c == 0 else term
            B.call("ff_ax_plus_y", B.ptr(factor), values, _vp(s["witness"][c]), into, n, stream)
            B.call("ff_a_plus_x", B.ptr(s["gamma"]), into, into, n, stream)
            if c:
                B.call("ff_x_mul_y", side, term, side, n, stream)
    B.call("ff_inverse", B.ff_inverse_configuration(_pool, stream, s["denominator"].data_ptr(), s["inverse"].data_ptr(), s["count"]))
    B.call("ff_x_mul_y", num, inv, _vp(s["ratio"]), n, stream)
    B.call("ff_grand_product", B.ff_grand_product_configuration(_pool, stream, s["ratio"].data_ptr(), s["z"].data_ptr(), s["count"]))
    return {"inverse": s["inverse"], "z": s["z"]}


def _run_opening(s, stream):
    """p_i(z) for every polynomial, sum_i v^i p_i, and that polynomial with its variable scaled by z."""
    n, z = s["count"], s["z"].ctypes.data
    combined = _vp(s["combined"])
    for i, poly in enumerate(s["polys"]):
        B.call("ff_poly_evaluate", B.ff_poly_evaluate_configuration(_pool, stream, poly.data_ptr(), z, s["evaluations"][i].data_ptr(), n))
    B.call("ff_ax_plus_y", B.ptr(s["v_powers"][1]), _vp(s["polys"][1]), _vp(s["polys"][0]), combined, _u(n), stream)
    for i in range(2, len(s["polys"])):
        B.call("ff_ax_plus_y", B.ptr(s["v_powers"][i]), _vp(s["polys"][i]), combined, combined, _u(n), stream)
    B.call("ff_multiply_by_powers", B.ff_multiply_by_powers_configuration(_pool, stream, s["combined"].data_ptr(), z, s["scaled"].data_ptr(), n))
    return {"evaluations": s["evaluations"], "combined": s["combined"], "scaled": s["scaled"]}


# ---------------------------------------------------------------- what a pass cannot do without
def _ntt_work(log_n):
    n = 1 << log_n
    return 64 * n, n * log_n // 2 * PRODUCT_OPS


def _msm_work(log_n):
    n = 1 << log_n
    windows = -(-254 // max(log_n - 3, 4))
    return 96 * n + 64, 10 * n * windows * PRODUCT_OPS


def work(case):
    kind = case["kind"]
    if kind == "ntt":
        nbytes, ops = _ntt_work(case["log_n"])
        ops += PRODUCT_OPS << case["log_n"] if case["log_ext"] else 0
    elif kind == "lde":
        one, ops = _ntt_work(case["log_n"])
        cosets = 1 << case["log_ext"]
        # values in, coefficients and every coset out
        nbytes, ops = one // 2 * (2 + cosets), ops * (1 + cosets) + (cosets * PRODUCT_OPS << case["log_n"])
    elif kind == "msm":
        nbytes, ops = _msm_work(case["log_n"])
    elif kind == "pn":
        cells = case["columns"] << case["log_rows"]
        nbytes, ops = 36 * cells, cells * PRODUCT_OPS
    elif kind == "copy_permutation":
        n, k = case["count"], case["columns"]
        # witness and sigma in, the inverse and z out; 2k scalings, 2(k - 1) products, 3 for an inverse, the ratio, the prefix
        nbytes, ops = 32 * n * (2 * k + 2), n * (2 * k + 2 * (k - 1) + 5) * PRODUCT_OPS
    elif kind == "opening":
        n, k = case["count"], case["polys"]
        nbytes, ops = 32 * n * (k + 2), n * (2 * k + 1) * PRODUCT_OPS
    else:
        parts = [_msm_work(l) for l in _spread(case["msm_log_min"], case["msm_log_max"], case["msms"])]
        parts += [_ntt_work(l) for l in _spread(case["ntt_log_min"], case["ntt_log_max"], case["ntts"])]
        nbytes, ops = sum(p[0] for p in parts), sum(p[1] for p in parts)
    return {"bytes": nbytes, "flops": ops}


# ---------------------------------------------------------------- the same in Python integers
def _ints(tensor):
    data = tensor.detach().cpu().contiguous().numpy().tobytes()
    return [int.from_bytes(data[i:i + 32], "little") for i in range(0, len(data), 32)]


def _tensor(values, *shape):
    return torch.from_numpy(_limbs(values).view(np.int32)).reshape(shape + (8,))


def _bit_reversed(values):
    log_n = (len(values) - 1).bit_length()
    index = np.zeros(len(values), dtype=np.int64)
    for b in range(log_n):
        index |= ((np.arange(len(values)) >> b) & 1) << (log_n - 1 - b)
    return values[index]


def _powers(base, count, first=1):
    out = np.empty(count, dtype=object)
    x = first
    for i in range(count):
        out[i] = x
        x = x * base % R
    return out


def _transform(values, inverse):
    """Natural order to natural order, by decimation in frequency and a bit reversal."""
    x = np.array(values, dtype=object)
    n = len(x)
    root = pow(ROOT_2_28, (1 << 28) // n, R)
    if inverse:
        root = pow(root, -1, R)
    size = n
    while size > 1:
        half = size // 2
        twiddles = _powers(pow(root, n // size, R), half)
        blocks = x.reshape(-1, size)
        low, high = blocks[:, :half].copy(), blocks[:, half:].copy()
        blocks[:, :half] = (low + high) % R
        blocks[:, half:] = (low - high) * twiddles % R
        size = half
    x = _bit_reversed(x)
    return x * pow(n, -1, R) % R if inverse else x


def _exact_ntt(values, log_n, bit_reversed, inverse, log_ext, coset):
    x = np.array(values, dtype=object)
    if bit_reversed:
        x = _bit_reversed(x)
    shift = GENERATOR * pow(pow(ROOT_2_28, 1 << (28 - log_n - log_ext), R), coset, R) % R if log_ext else 1
    if log_ext and not inverse:
        x = x * _powers(shift, len(x)) % R
    y = _transform(x, inverse)
    if log_ext and inverse:
        y = y * _powers(pow(shift, -1, R), len(y)) % R
    return y if bit_reversed else _bit_reversed(y)


def _add_points(a, b):
    if a is None or b is None:
        return a or b
    if a[0] == b[0]:
        if (a[1] + b[1]) % P == 0:
            return None
        slope = 3 * a[0] * a[0] * pow(2 * a[1], -1, P) % P
    else:
        slope = (b[1] - a[1]) * pow(b[0] - a[0], -1, P) % P
    x = (slope * slope - a[0] - b[0]) % P
    return x, (slope * (a[0] - x) - a[1]) % P


def _commitment(scalars, logs):
    """[sum k s] G as affine Montgomery coordinates, (0, 0) for infinity."""
    k = sum(a * b for a, b in zip(scalars, logs)) % R
    total, double = None, (1, 2)
    while k:
        if k & 1:
            total = _add_points(total, double)
        double = _add_points(double, double)
        k >>= 1
    x, y = total or (0, 0)
    return torch.from_numpy(_limbs([x * MONT % P, y * MONT % P]).view(np.int32)).reshape(1, 16)


def exact(case, seed):
    kind = case["kind"]
    # butterflies, terms or cells that about 20 seconds of Python allow
    if kind in ("ntt", "lde"):
        transforms = 1 if kind == "ntt" else 1 + (1 << case["log_ext"])
        if transforms * case["log_n"] << case["log_n"] > 1 << 24:
            return None
    elif kind == "msm" and case["log_n"] > 21:
        return None
    elif kind == "pn" and case["columns"] << case["log_rows"] > 1 << 22:
        return None
    elif kind in ("copy_permutation", "opening") and case["count"] * (3 * case.get("columns", case.get("polys"))) > 1 << 24:
        return None
    elif kind == "batch" and (case["msms"] << case["msm_log_max"]) + 10 * (case["ntts"] << case["ntt_log_max"]) > 1 << 26:
        return None
    _library()
    x = _inputs(case, seed)
    unmont = pow(MONT, -1, R)
    if kind == "ntt":
        y = _exact_ntt(_ints(x["values"]), case["log_n"], case["bit_reversed"], case["inverse"], case["log_ext"], case["coset"])
        return _tensor(y, len(y))
    if kind == "lde":
        coefficients = _transform(_ints(x["values"]), True)
        cosets = [_exact_ntt(coefficients, case["log_n"], False, False, case["log_ext"], c) for c in range(1 << case["log_ext"])]
        n = len(coefficients)
        return {"coefficients": _tensor(coefficients, n), "cosets": _tensor(np.concatenate(cosets), len(cosets), n)}
    if kind == "msm":
        return _commitment(_ints(x["scalars"]), _ints(x["logs"]))
    if kind == "pn":
        return _exact_pn(case, x)
    if kind == "copy_permutation":
        n, k = case["count"], case["columns"]
        beta, gamma = x["challenges"][:2]
        shifts = [1] + x["challenges"][2:2 + k - 1]
        domain = _powers(pow(ROOT_2_28, 1 << (28 - max(n - 1, 1).bit_length()), R), n)
        num = den = 1
        for c in range(k):
            w, sigma = (np.array(_ints(t[c]), dtype=object) * unmont % R for t in (x["witness"], x["sigma"]))
            num = num * ((w + beta * shifts[c] * domain + gamma) % R) % R
            den = den * ((w + beta * sigma + gamma) % R) % R
        inverse = [pow(d, -1, R) if d else 0 for d in den]
        z, total = [], 1
        for a, b in zip(num, inverse):
            total = total * a * b % R
            z.append(total * MONT % R)
        return {"inverse": _tensor([v * MONT % R for v in inverse], n), "z": _tensor(z, n)}
    if kind == "opening":
        n = case["count"]
        z, v = x["challenges"]
        powers = _powers(z, n)
        polys = [np.array(_ints(p), dtype=object) for p in x["polys"]]
        combined = sum(p * pow(v, i, R) for i, p in enumerate(polys)) % R
        return {"evaluations": _tensor([int((p * powers).sum()) % R for p in polys], len(polys)), "combined": _tensor(combined, n),
                "scaled": _tensor(combined * powers % R, n)}
    logs = _ints(x["logs"])
    return {"points": torch.cat([_commitment(_ints(s), logs) for s in x["scalars"]]),
            "transforms": [_tensor(_exact_ntt(_ints(v), l, False, False, 0, 0), 1 << l) for v, l in zip(x["values"], x["ntt_logs"])]}


def _exact_pn(case, x):
    """Each cell takes the identity value of the next cell of its cycle in
    row-major order; the cycle of the smallest variable keeps the identity."""
    rows, cols = 1 << case["log_rows"], case["columns"]
    omega = _powers(pow(ROOT_2_28, (1 << 28) // rows, R), rows)
    identity = np.concatenate([omega * f % R for f in _ints(x["factors"])])
    keys = x["indexes"].cpu().numpy().view(np.uint32).reshape(cols, rows).T.reshape(-1)
    cell = (np.arange(cols)[None, :] * rows + np.arange(rows)[:, None]).reshape(-1)
    order = np.argsort(keys, kind="stable")
    keys, cell = keys[order], cell[order]
    starts = np.flatnonzero(np.concatenate([[True], keys[1:] != keys[:-1]]))
    ends = np.concatenate([starts[1:], [len(keys)]])
    source = np.arange(len(keys)) + 1
    source[ends - 1] = starts
    source[:ends[0]] = np.arange(ends[0])
    out = np.empty(len(keys), dtype=object)
    out[cell] = identity[cell[source]]
    return _tensor(out, cols, rows)
