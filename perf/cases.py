"""Timing cases of the prover hot path, each one pass through the public operators.

A case is what a prover does between two instructions of its program: a transform
over a resident polynomial, a commitment, a grand product, an opening, a lookup
permutation, the fused gate expressions, or a batch of those in one graph launch.
Every result is exact field or group arithmetic, so outputs are whole numbers
(64-bit limbs, Montgomery form) and any correct implementation gives the same bytes.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "zkpoly-compiler_amd"))

from zkpoly_amd import batch, fused, hip, msm, ntt, poly  # noqa: E402
from zkpoly_amd.runtime import (  # noqa: E402
    GpuBuffer,
    Libs,
    Point,
    PointArray,
    PolyPtr,
    Scalar,
    ScalarArray,
)

R = 0x30644E72E131A029B85045B68181585D2833E84879B9709143E1F593F0000001  # scalar field
Q = 0x30644E72E131A029B85045B68181585D97816A916871CA8D3C208C16D87CFD47  # base field
MONT = 1 << 256
MONT_INV = pow(MONT, -1, R)
ROOT_2_28 = 0x03DDB9F5166D18B798865EA93DD31F743215CF6DD39329C8D34F1ED960C37C9C  # order 2^28
ZETA = pow(7, (R - 1) // 3, R)  # the extended domain's coset element (order 3)
TOP_LIMB = 0x30644E72E131A029  # random top limbs stay below it, so values stay below R
MAC = 136  # 32 x 32-bit multiply-adds of one Montgomery product
CUDA = "cuda:0"


# ---------------------------------------------------------------- cases

def listed():
    return [
        # a small column's transform: two launches, nearly all latency
        {"name": "ntt_12", "kind": "ntt", "log_n": 12, "rotate": 0},
        # Lagrange to coefficients of a 2^20-row circuit's column (inverse root, then 1/n)
        {"name": "intt_20", "kind": "intt", "log_n": 20, "rotate": 0},
        # a column of coefficients onto the four times larger coset domain of the quotient
        {"name": "extend_22", "kind": "extend", "log_n": 20},
        # the largest transform of the benchmark, the whole chip on one polynomial
        {"name": "ntt_24", "kind": "ntt", "log_n": 24, "rotate": 0},
        # the transform whose twiddle table does not fit beside the proof's other constants
        {"name": "recompute_21", "kind": "recompute", "log_n": 21, "rotate": 0},
        # commitment to a column with resident bases and scalars
        {"name": "msm_device_20", "kind": "msm", "n": 1 << 20, "window": 16, "ones": 0},
        # drop-in commitment of witness columns (a tenth zeros, a tenth ones) from pinned host memory
        {"name": "msm_host_17", "kind": "msm_host", "n": 150001, "window": 13, "tables": 1, "batches": 2, "parts": 1,
         "ones": 1},
        # one proof step of many uneven transforms, their gate expression and commitments in one graph launch
        {"name": "step_24", "kind": "step", "count": 24, "lo": 10, "hi": 18, "msms": 6, "msm_lo": 10, "msm_hi": 14},
        # a permutation argument's running product over the usable rows
        {"name": "product_20", "kind": "product", "n": (1 << 20) - 6, "zeros": 0},
        # opening of a polynomial at one point: its value and the quotient
        {"name": "opening_21", "kind": "opening", "log_n": 21},
        # lookup argument over the usable rows, compressed expressions, repeated values
        {"name": "lookup_20", "kind": "lookup", "n": (1 << 20) - 6, "distinct": 1 << 18},
        # the constraint expressions of a circuit fused into one kernel of 800 vertices
        {"name": "gates_18", "kind": "gates", "n": 1 << 18, "graph": "large"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ntt", "intt", "extend", "recompute", "msm", "msm_host", "step", "product", "opening",
                       "lookup", "gates"])
    if kind in ("ntt", "intt", "recompute"):
        k = rng.randint(10, {"ntt": 23, "intt": 23, "recompute": 22}[kind])
        # a polynomial read at a rotation is transformed in place through its rotated view
        return {"kind": kind, "log_n": k, "rotate": rng.choice([0, rng.randrange(1, 1 << k)])}
    if kind == "extend":
        return {"kind": kind, "log_n": rng.randint(8, 20)}
    if kind == "msm":
        n = _log_uniform(rng, 1 << 11, 1 << 20)
        return {"kind": kind, "n": n, "window": batch.default_msm_window(n.bit_length() - 1),
                "ones": rng.randint(0, 1)}
    if kind == "msm_host":
        n = _log_uniform(rng, 1 << 14, 1 << 18)
        tables = rng.randint(1, 2)
        return {"kind": kind, "n": n, "window": rng.randint(12, 15), "tables": tables,
                "batches": rng.randint(1, 3), "parts": rng.randint(1, 2), "ones": rng.randint(0, 1)}
    if kind == "step":
        lo = rng.randint(8, 12)
        return {"kind": kind, "count": rng.randint(4, 24), "lo": lo, "hi": rng.randint(lo + 2, 18),
                "msms": rng.randint(1, 6), "msm_lo": 10, "msm_hi": rng.randint(11, 14)}
    if kind == "product":
        return {"kind": kind, "n": _log_uniform(rng, 1 << 10, 1 << 22), "zeros": rng.randint(0, 1)}
    if kind == "opening":
        return {"kind": kind, "log_n": rng.randint(10, 22)}
    if kind == "lookup":
        n = _log_uniform(rng, 1 << 12, 1 << 21)
        return {"kind": kind, "n": n, "distinct": _log_uniform(rng, 16, n)}
    return {"kind": kind, "n": _log_uniform(rng, 1 << 11, 1 << 19), "graph": rng.choice(["large", "abgcz"])}


# ---------------------------------------------------------------- inputs

_CONTEXT = {}


def _context():
    """The libraries and the stream that a program holds for its lifetime."""
    if not _CONTEXT:
        torch.cuda.init()
        _CONTEXT["libs"] = Libs()
        _CONTEXT["stream"] = hip.Stream(0)
    return _CONTEXT["libs"], _CONTEXT["stream"]


def _generator(seed, salt=0, device=CUDA):
    return torch.Generator(device=device).manual_seed(seed * 1000003 + salt)


def _elements(n, gen):
    """n field elements, limbs (n, 4), every bit of the lower limbs and all top limbs below R's."""
    x = torch.randint(-(1 << 63), (1 << 63) - 1, (n, 4), dtype=torch.int64, device=CUDA, generator=gen)
    x[:, 3] = torch.randint(0, TOP_LIMB, (n,), dtype=torch.int64, device=CUDA, generator=gen)
    return x


def _limbs(x):
    return [((x >> (64 * i)) & ((1 << 64) - 1)) - ((((x >> (64 * i)) >> 63) & 1) << 64) for i in range(4)]


def _constant(x):
    """A canonical value as one resident Montgomery element."""
    return torch.tensor([_limbs(x * MONT % R)], dtype=torch.int64, device=CUDA)


def _array(t, rotate=0):
    a = ScalarArray(t.shape[0], t.data_ptr())
    if rotate:
        a.rotate(rotate)
    return a


def _temp(nbytes):
    t = torch.empty(max(int(nbytes), 16), dtype=torch.uint8, device=CUDA)
    return t, GpuBuffer(t.data_ptr(), int(nbytes))


def _omega(k, inverse=False):
    w = pow(ROOT_2_28, 1 << (28 - k), R)
    return pow(w, -1, R) if inverse else w


def _twiddles(k, inverse=False):
    libs, stream = _context()
    tw = torch.empty(((1 << k) // 2, 4), dtype=torch.int64, device=CUDA)
    w = _constant(_omega(k, inverse))
    torch.cuda.synchronize()
    ntt.gen_powers(libs, tw.data_ptr(), tw.shape[0], w.data_ptr(), stream)
    stream.sync()
    return tw


def _witness(n, seed, salt, ones):
    """Scalars of one column; with `ones` a tenth of them 0 and a tenth 1, as witnesses have."""
    gen = _generator(seed, salt)
    s = _elements(n, gen)
    if ones:
        u = torch.rand(n, device=CUDA, generator=gen)
        s[u < 0.1] = 0
        s[(u >= 0.1) & (u < 0.2)] = _constant(1)[0]
    return s


def _bases(n, seed):
    """P_i = k_i G for seeded k_i, affine (n, 8), resident."""
    libs, stream = _context()
    k = _elements(n, _generator(seed, 77))
    p = torch.empty((n, 8), dtype=torch.int64, device=CUDA)
    torch.cuda.synchronize()
    msm.mul_generator(libs, k.data_ptr(), n, p.data_ptr(), stream)
    stream.sync()
    return p


def _fused_kernel(name, num_vars, num_mut, lib_dir):
    libs, _ = _context()
    return fused.FusedKernel(libs, fused.FusedKernelMeta(name, num_vars, num_mut, lib_dir))


def _step_logs(case):
    span = case["hi"] - case["lo"] + 1
    mspan = case["msm_hi"] - case["msm_lo"] + 1
    return ([case["lo"] + (5 * i + i // span) % span for i in range(case["count"])],
            [case["msm_lo"] + (3 * i) % mspan for i in range(case["msms"])])


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    libs, stream = _context()
    s = {"case": dict(case), "stream": stream}
    globals()["_prepare_" + case["kind"]](case, seed, libs, stream, s)
    torch.cuda.synchronize()
    return s


def _prepare_ntt(case, seed, libs, stream, s):
    s["x"] = _elements(1 << case["log_n"], _generator(seed))
    s["tw"] = _twiddles(case["log_n"])
    s["args"] = ([_array(s["x"], case["rotate"])], [_array(s["tw"]), stream])
    s["ntt"] = ntt.SsipNtt(libs).get_fn().f


def _prepare_intt(case, seed, libs, stream, s):
    k = case["log_n"]
    s["x"] = _elements(1 << k, _generator(seed))
    s["tw"] = _twiddles(k, inverse=True)
    s["scale"] = _constant(pow(1 << k, -1, R))
    s["poly"] = _array(s["x"], case["rotate"])
    s["ntt"] = ntt.SsipNtt(libs).get_fn().f
    s["distribute"] = ntt.DistributePowers(libs).get_fn().f


def _prepare_extend(case, seed, libs, stream, s):
    n = 1 << case["log_n"]
    s["coef"] = _elements(n, _generator(seed))
    s["out"] = torch.empty((4 * n, 4), dtype=torch.int64, device=CUDA)
    s["tw"] = _twiddles(case["log_n"] + 2)
    s["zeta"] = torch.cat([_constant(pow(ZETA, i, R)) for i in range(3)])
    s["ntt"] = ntt.SsipNtt(libs).get_fn().f
    s["distribute"] = ntt.DistributePowers(libs).get_fn().f
    s["zero"] = poly.PolyZero(libs).get_fn().f
    s["add"] = poly.PolyAdd(libs).get_fn().f


def _prepare_recompute(case, seed, libs, stream, s):
    k = case["log_n"]
    s["x"] = _elements(1 << k, _generator(seed))
    gen = ntt.GenPqOmegas(libs)
    pq = np.zeros((gen.get_pq_len(k), 4), dtype=np.uint64)
    ladder = np.zeros((32, 4), dtype=np.uint64)
    unit = np.array(_limbs(_omega(k) * MONT % R), dtype=np.int64).view(np.uint64)
    gen.get_fn()(ScalarArray(len(pq), pq.ctypes.data, "cpu"), ScalarArray(32, ladder.ctypes.data, "cpu"), 1 << k, unit)
    s["pq"] = torch.from_numpy(pq.view(np.int64)).to(CUDA)
    s["ladder"] = torch.from_numpy(ladder.view(np.int64)).to(CUDA)
    s["args"] = ([_array(s["x"], case["rotate"])], [_array(s["pq"]), _array(s["ladder"]), stream])
    s["ntt"] = ntt.RecomputeNtt(libs).get_fn().f


def _prepare_msm(case, seed, libs, stream, s):
    n, w = case["n"], case["window"]
    s["points"] = _bases(n, seed)
    s["scalars"] = _witness(n, seed, 1, case["ones"])
    s["target"] = -(-254 // w)
    s["workspace"] = hip.DeviceBuffer(msm.workspace_size(libs, n, w, s["target"]))
    s["libs"] = libs


def _prepare_msm_host(case, seed, libs, stream, s):
    n, windows = case["n"], -(-254 // case["window"])
    cfg = msm.MsmConfig(case["window"], -(-windows // case["tables"]), batch_per_run=case["batches"],
                        parts=case["parts"], stage_scalars=2, stage_points=min(2, case["parts"]))
    s["tables"] = [torch.empty((n, 8), dtype=torch.int64, pin_memory=True) for _ in range(cfg.get_precompute())]
    s["tables"][0].copy_(_bases(n, seed))
    points = [PointArray(t.data_ptr(), n) for t in s["tables"]]
    if len(points) > 1:
        msm.MSMPrecompute(libs, cfg).get_fn()(points, n, 1)
    s["scalars"] = []
    for b in range(case["batches"]):
        t = torch.empty((n, 4), dtype=torch.int64, pin_memory=True)
        t.copy_(_witness(n, seed, 1 + b, case["ones"]))
        s["scalars"].append(t)
    op = msm.MSM(libs, cfg)
    s["temp"], buffer = _temp(op.get_buffer_size(n)[0])
    s["results"] = [Point() for _ in range(case["batches"])]
    s["args"] = ([buffer] + s["results"], points + [ScalarArray(n, t.data_ptr(), "cpu") for t in s["scalars"]])
    s["msm"] = op.get_fn().f


def _prepare_step(case, seed, libs, stream, s):
    logs, msm_logs = _step_logs(case)
    lens = [1 << k for k in logs]
    starts = [sum(lens[:i]) for i in range(len(lens))]
    s["x"], s["out"] = _elements(sum(lens), _generator(seed)), torch.empty((sum(lens), 4), dtype=torch.int64, device=CUDA)
    s["abc"] = [_elements(sum(lens), _generator(seed, 2 + j)) for j in range(3)]
    s["gz"] = _elements(2, _generator(seed, 5))
    s["tw"] = {k: _twiddles(k) for k in sorted(set(logs))}

    def views(t):
        return [PolyPtr(t.data_ptr() + 32 * a, n, 0, 0, n) for a, n in zip(starts, lens)]

    gamma, z = (PolyPtr(s["gz"].data_ptr() + 32 * i, 1, 0, 0, 1) for i in range(2))
    columns = [views(t) for t in s["abc"]]
    kernel = _fused_kernel("fused_arith_abgcz", 5, 1, fused.DEMO_DIR)
    vars_ = [v for i in range(len(lens)) for v in (columns[0][i], columns[1][i], columns[2][i], gamma, z)]
    s["points"] = _bases(1 << max(msm_logs), seed)
    s["scalars"] = [_witness(1 << k, seed, 10 + j, j % 2) for j, k in enumerate(msm_logs)]
    torch.cuda.synchronize()
    msms = [msm.DeviceMsm(libs, s["points"].data_ptr(), t.data_ptr(), t.shape[0], batch.default_msm_window(k))
            for t, k in zip(s["scalars"], msm_logs)]
    for m in msms:  # the first MSM on a device sets its launch limits, before any capture
        m.enqueue(stream)
    stream.sync()
    transforms = batch.NttBatch(libs, views(s["x"]), [s["tw"][k].data_ptr() for k in logs], logs)
    s["step"] = batch.ProofStepBatch(stream, transforms, batch.FusedBatch(kernel, vars_, views(s["out"]), lens), msms)


def _prepare_product(case, seed, libs, stream, s):
    n = case["n"]
    s["num"], s["den0"] = (_elements(n, _generator(seed, j)) for j in range(2))
    if case["zeros"]:  # rows whose denominator is zero keep a zero
        s["den0"][torch.rand(n, device=CUDA, generator=_generator(seed, 9)) < 0.01] = 0
        s["den0"][0] = _constant(1)[0]
    s["den"], s["ratio"], s["z"] = (torch.empty_like(s["num"]) for _ in range(3))
    s["one"] = _constant(1)
    invert, scan = poly.PolyInvert(libs), poly.PolyScan(libs)
    s["t1"], s["invert_temp"] = _temp(invert.get_buffer_size(n))
    s["t2"], s["scan_temp"] = _temp(scan.get_buffer_size(n))
    s["copy"] = poly.PolyAdd(libs).get_fn().f
    s["mul"] = poly.PolyMul(libs).get_fn().f
    s["invert"], s["scan"] = invert.get_fn().f, scan.get_fn().f


def _prepare_opening(case, seed, libs, stream, s):
    n = 1 << case["log_n"]
    s["p"] = _elements(n, _generator(seed))
    s["x"] = _elements(1, _generator(seed, 1))
    s["q"], s["value"] = torch.empty_like(s["p"]), torch.empty((1, 4), dtype=torch.int64, device=CUDA)
    evaluate, kate = poly.PolyEval(libs), poly.KateDivision(libs)
    s["t1"], s["eval_temp"] = _temp(evaluate.get_buffer_size(n))
    s["t2"], s["kate_temp"] = _temp(kate.get_buffer_size(case["log_n"]))
    s["eval"], s["kate"] = evaluate.get_fn().f, kate.get_fn().f


def _lookup_rows(case, seed):
    n, distinct = case["n"], case["distinct"]
    gen = _generator(seed)
    values = _elements(distinct, gen)
    table = values[torch.randint(0, distinct, (n,), device=CUDA, generator=gen)]
    table[:distinct] = values
    rows = values[torch.randint(0, distinct, (n,), device=CUDA, generator=gen)]
    return rows, table[torch.randperm(n, device=CUDA, generator=gen)].contiguous()


def _prepare_lookup(case, seed, libs, stream, s):
    s["input"], s["table"] = _lookup_rows(case, seed)
    s["res_input"], s["res_table"] = torch.empty_like(s["input"]), torch.empty_like(s["table"])
    op = poly.PolyPermute(libs)
    s["t"], s["temp"] = _temp(op.get_buffer_size(case["n"]))
    s["permute"] = op.get_fn().f


def _prepare_gates(case, seed, libs, stream, s):
    n = case["n"]
    if case["graph"] == "large":
        kernel = _fused_kernel(fused.large_kernel_name(fused.LARGE_SEEDS[0], False), 18, 21, fused.LARGE_DIR)
        polys, scalars, outs, scalar_outs = 12, 6, 18, 3
    else:
        kernel = _fused_kernel("fused_arith_abgcz", 5, 1, fused.DEMO_DIR)
        polys, scalars, outs, scalar_outs = 3, 2, 1, 0
    s["in"] = [_elements(n, _generator(seed, j)) for j in range(polys)]
    s["scalars"] = _elements(scalars, _generator(seed, 100))
    # the first two outputs of the large graph overwrite inputs of the same place
    s["out"] = [_elements(n, _generator(seed, 50 + j)) for j in range(outs)]
    s["scalar_out"] = torch.zeros((max(scalar_outs, 1), 4), dtype=torch.int64, device=CUDA)
    s["arg"], arg = _temp(fused.arg_buffer_bytes(kernel.meta))
    s["local"], local = _temp(kernel.local_bytes)
    s["vars"] = [stream] + [_array(t) for t in s["in"]] + [Scalar(s["scalars"].data_ptr() + 32 * j)
                                                           for j in range(scalars)]
    s["muts"] = [arg, local] + [_array(t) for t in s["out"]] + [Scalar(s["scalar_out"].data_ptr() + 32 * j)
                                                                for j in range(scalar_outs)]
    s["fused"] = kernel.get_fn().f


# ---------------------------------------------------------------- run

def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _run_ntt(s):
    s["ntt"](*s["args"])
    return s["x"]


def _run_intt(s):
    s["ntt"]([s["poly"]], [_array(s["tw"]), s["stream"]])
    s["distribute"]([s["poly"]], [_array(s["scale"]), s["stream"]])
    return s["x"]


def _run_extend(s):
    out, coef = _array(s["out"]), _array(s["coef"])
    n = coef.len
    s["zero"]([out.slice(n, 4 * n)], [s["stream"]])
    head = out.slice(0, n)
    s["add"]([head], [coef, ScalarArray(0, 0), s["stream"]])
    s["distribute"]([head], [_array(s["zeta"]), s["stream"]])
    s["ntt"]([out], [_array(s["tw"]), s["stream"]])
    return s["out"]


def _run_recompute(s):
    s["ntt"](*s["args"])
    return s["x"]


def _run_msm(s):
    c = s["case"]
    got = msm.msm_device(s["libs"], s["points"].data_ptr(), s["scalars"].data_ptr(), c["n"], c["window"], s["target"],
                         s["workspace"], s["stream"])
    return got.view(np.int64)


def _run_msm_host(s):
    s["msm"](*s["args"])
    return np.stack([p.data for p in s["results"]]).view(np.int64)


def _run_step(s):
    s["step"].launch(s["stream"])
    s["stream"].sync()
    return [s["x"], s["out"], np.stack(s["step"].msm_results()).view(np.int64)]


def _run_product(s):
    stream = s["stream"]
    num, den, ratio, z = (_array(s[k]) for k in ("num", "den", "ratio", "z"))
    s["copy"]([den], [_array(s["den0"]), ScalarArray(0, 0), stream])
    s["invert"]([s["invert_temp"], den], [stream])
    s["mul"]([ratio], [num, den, stream])
    s["scan"]([s["scan_temp"], z], [ratio, Scalar(s["one"].data_ptr()), stream])
    return [s["den"], s["z"]]


def _run_opening(s):
    p, x = _array(s["p"]), Scalar(s["x"].data_ptr())
    s["eval"]([s["eval_temp"], Scalar(s["value"].data_ptr())], [p, x, s["stream"]])
    s["kate"]([s["kate_temp"], _array(s["q"])], [p, x, s["stream"]])
    return [s["value"], s["q"]]


def _run_lookup(s):
    s["permute"]([_array(s["res_input"]), _array(s["res_table"]), s["temp"]],
                 [_array(s["input"]), _array(s["table"]), s["stream"]])
    return [s["res_input"], s["res_table"]]


def _run_gates(s):
    s["fused"](s["muts"], s["vars"])
    return s["out"] + [s["scalar_out"]]


# ---------------------------------------------------------------- work and tolerance

def _ntt_work(n, products):
    """In and out once (twiddles are the plan's); the butterflies' products and `products` more."""
    return {"bytes": 64 * n, "flops": 2 * MAC * (n // 2 * (n.bit_length() - 1) + products)}


def _msm_work(n, window, batches=1):
    """Ten products for each point's signed digit, 28 for each bucket; points and scalars once."""
    windows = -(-254 // window)
    products = batches * windows * (10 * n + 28 * (1 << (window - 1)))
    return {"bytes": (64 + 32 * batches) * n, "flops": 2 * MAC * products}


def work(case):
    kind = case["kind"]
    if kind in ("ntt", "recompute"):
        return _ntt_work(1 << case["log_n"], 0)
    if kind == "intt":
        return _ntt_work(1 << case["log_n"], 1 << case["log_n"])
    if kind == "extend":
        n = 4 << case["log_n"]
        return dict(_ntt_work(n, n // 4), bytes=40 * n)
    if kind == "msm":
        return _msm_work(case["n"], case["window"])
    if kind == "msm_host":
        return _msm_work(case["n"], case["window"], case["batches"])
    if kind == "step":
        logs, msm_logs = _step_logs(case)
        parts = [_ntt_work(1 << k, 0) for k in logs]
        parts += [{"bytes": 128 << k, "flops": 2 * MAC * (2 << k)} for k in logs]
        parts += [_msm_work(1 << k, batch.default_msm_window(k)) for k in msm_logs]
        return {key: sum(p[key] for p in parts) for key in ("bytes", "flops")}
    if kind == "product":
        # numerators and denominators in; inverses (three products each) and running products out
        return {"bytes": 128 * case["n"], "flops": 2 * MAC * 5 * case["n"]}
    if kind == "opening":
        return {"bytes": 64 << case["log_n"], "flops": 2 * MAC * (2 << case["log_n"])}
    if kind == "lookup":
        return {"bytes": 128 * case["n"], "flops": 0}
    if case["graph"] == "large":
        # 14 columns in, 18 out; about 340 products and powers of an element
        return {"bytes": 32 * 32 * case["n"], "flops": 2 * MAC * 340 * case["n"]}
    return {"bytes": 128 * case["n"], "flops": 2 * MAC * 2 * case["n"]}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------- exact values (integers, no code of the package)

def _ints(t):
    a = t.cpu().numpy().view(np.uint64).astype(object)
    return list(a[:, 0] + (a[:, 1] << 64) + (a[:, 2] << 128) + (a[:, 3] << 192))


def _tensor(values):
    return torch.tensor([_limbs(v) for v in values], dtype=torch.int64)


def _transform(values, w):
    """Natural-order DFT of a power-of-two list by halves."""
    n = len(values)
    if n == 1:
        return values
    even, odd = _transform(values[0::2], w * w % R), _transform(values[1::2], w * w % R)
    out, f = [0] * n, 1
    for i in range(n // 2):
        t = odd[i] * f % R
        out[i], out[i + n // 2] = (even[i] + t) % R, (even[i] - t) % R
        f = f * w % R
    return out


def _point_add(a, b):
    if a is None or b is None:
        return b if a is None else a
    if a[0] == b[0]:
        if (a[1] + b[1]) % Q == 0:
            return None
        m = 3 * a[0] * a[0] * pow(2 * a[1], -1, Q) % Q
    else:
        m = (b[1] - a[1]) * pow(b[0] - a[0], -1, Q) % Q
    x = (m * m - a[0] - b[0]) % Q
    return x, (m * (a[0] - x) - a[1]) % Q


def _commitment(n, seed, salt, ones):
    """(sum of k_i s_i) G as the affine result's eight limbs."""
    k, s = _ints(_elements(n, _generator(seed, 77))), _ints(_witness(n, seed, salt, ones))
    e = sum(a * b for a, b in zip(k, s)) * MONT_INV * MONT_INV % R
    acc, base = None, (1, 2)
    while e:
        if e & 1:
            acc = _point_add(acc, base)
        base, e = _point_add(base, base), e >> 1
    x, y = acc or (0, 0)
    return _limbs(x * MONT % Q) + _limbs(y * MONT % Q)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("ntt", "intt", "recompute", "extend"):
        if case["log_n"] > 15:
            return None
        k = case["log_n"]
        values = _ints(_elements(1 << k, _generator(seed)))
        if kind == "extend":
            values = [v * pow(ZETA, i % 3, R) % R for i, v in enumerate(values)] + [0] * (3 << k)
            return _tensor(_transform(values, _omega(k + 2)))
        r = case["rotate"]  # the view's element i is the array's element (i - r) mod n
        n = 1 << k
        out = _transform([values[(i - r) % n] for i in range(n)], _omega(k, kind == "intt"))
        if kind == "intt":
            scale = pow(n, -1, R)
            out = [v * scale % R for v in out]
        return _tensor([out[(i + r) % n] for i in range(n)])
    if kind == "msm":
        return np.array(_commitment(case["n"], seed, 1, case["ones"]), dtype=np.int64)
    if kind == "msm_host":
        return np.array([_commitment(case["n"], seed, 1 + b, case["ones"]) for b in range(case["batches"])],
                        dtype=np.int64)
    if kind == "product":
        if case["n"] > 1 << 16:
            return None
        num, den = (_ints(_elements(case["n"], _generator(seed, j))) for j in range(2))
        if case["zeros"]:
            gone = (torch.rand(case["n"], device=CUDA, generator=_generator(seed, 9)) < 0.01).tolist()
            den = [0 if g else d for g, d in zip(gone, den)]
            den[0] = MONT % R
        inverse = [pow(d, -1, R) * MONT * MONT % R if d else 0 for d in den]
        z = [MONT % R]
        for a, b in zip(num[:-1], inverse):
            z.append(z[-1] * (a * b * MONT_INV % R) * MONT_INV % R)
        return [_tensor(inverse), _tensor(z)]
    if kind == "opening":
        if case["log_n"] > 20:
            return None
        p = _ints(_elements(1 << case["log_n"], _generator(seed)))
        x = _ints(_elements(1, _generator(seed, 1)))[0] * MONT_INV % R
        q, acc = [0] * len(p), 0
        for i in range(len(p) - 1, -1, -1):
            q[i], acc = acc, (acc * x + p[i]) % R
        return [_tensor([acc]), _tensor(q)]
    if kind == "lookup":
        rows, table = (sorted(v * MONT_INV % R for v in _ints(t)) for t in _lookup_rows(case, seed))
        fresh = [i == 0 or rows[i] != rows[i - 1] for i in range(len(rows))]
        used, rest = {v for v, f in zip(rows, fresh) if f}, []
        for v in table:  # one table row of each value used goes to its first row
            if v in used:
                used.remove(v)
            else:
                rest.append(v)
        rest = iter(rest)
        out = [v if f else next(rest) for v, f in zip(rows, fresh)]
        return [_tensor([v * MONT % R for v in rows]), _tensor([v * MONT % R for v in out])]
    if kind == "gates" and case["graph"] == "abgcz":
        a, b, c = (_ints(_elements(case["n"], _generator(seed, j))) for j in range(3))
        gamma, z = _ints(_elements(2, _generator(seed, 100)))
        out = [((x * y + gamma * w) * MONT_INV - z) % R for x, y, w in zip(a, b, c)]
        return [_tensor(out), None]
    return None
