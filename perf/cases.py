"""The calls whose speed counts: LU factor-and-solve through the package's
public entry points, from the smallest batch to one matrix that fills the
device.

Every system is a full matrix with entries U[-1, 1] and one entry larger by
sqrt(n) in each row and column, in no order (a Jacobian whose equations come
in any order): partial pivoting moves a row at nearly every step, and the
solution is well determined. The solvers overwrite their inputs, so a pass
first copies them to the buffers that it works on, as a program does that
keeps its matrix (to refine, to form residuals or to assemble the next one).

Storage is the package's: a batch of column-major matrices is a (batch,
columns, ld) tensor, one matrix a (columns, ld) tensor.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from magma_amd import autotune, dense, iteref
from magma_amd import batched as mb
from magma_amd._ffi import MagmaNoTrans, MagmaTrans
from magma_amd.autograd import solve

DTYPES = {"f64": torch.float64, "f32": torch.float32}


def listed():
    return [
        # many small systems in one call (element matrices, small reaction networks): the latency of a call
        {"name": "gesv_1000x32", "op": "gesv", "batch": 1000, "n": 32, "ld": 32, "nrhs": 1},
        # the benchmark's workload
        {"name": "gesv_20000x128_r4", "op": "gesv", "batch": 20000, "n": 128, "ld": 128, "nrhs": 4},
        # an odd order in a padded buffer
        {"name": "gesv_3000x77_ld80_r3", "op": "gesv", "batch": 3000, "n": 77, "ld": 80, "nrhs": 3},
        # the largest order of the benchmark's fixed-size batches
        {"name": "gesv_2000x256", "op": "gesv", "batch": 2000, "n": 256, "ld": 256, "nrhs": 1},
        # single precision, factor then solve
        {"name": "f32_1000x300_r8", "op": "factor_solve_f32", "batch": 1000, "n": 300, "ld": 300, "nrhs": 8},
        # kept factors, new right-hand sides: the transposed system
        {"name": "getrs_trans_1000x384_r16", "op": "getrs", "batch": 1000, "n": 384, "ld": 384, "nrhs": 16,
         "trans": True},
        # systems of mixed order, one replay of a captured plan (the benchmark's ranges)
        {"name": "vbatched_6000_8to512", "op": "vbatched", "batch": 6000, "nmin": 8, "nmax": 512, "rmax": 16},
        # a differentiable solve inside a training step, forward and backward
        {"name": "adjoint_f64_8192x64_r8", "op": "adjoint", "dtype": "f64", "batch": 8192, "n": 64, "nrhs": 8},
        {"name": "adjoint_f32_8192x64_r8", "op": "adjoint", "dtype": "f32", "batch": 8192, "n": 64, "nrhs": 8},
        # mixed precision on a batch: 16-bit update, FP64 refinement
        {"name": "iteref_2000x256_fp16", "op": "iteref_batched", "batch": 2000, "n": 256, "ld": 256, "nrhs": 1,
         "facto": "fp16", "solver": "ir"},
        # one large matrix in FP64
        {"name": "dense_10000", "op": "dense", "n": 10000, "nrhs": 1},
        # one large matrix in mixed precision (the benchmark's order), the solver's default modes
        {"name": "dense_iteref_24576_fp16", "op": "dense_iteref", "n": 24576, "nrhs": 1, "facto": "fp16",
         "solver": "gmres"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch_for(rng, n, elements):
    """A batch count, spread over its logarithm, of at most `elements` matrix entries."""
    return _log(rng, 1, max(2, min(50000, elements // (n * n))))


def draw(rng):
    op = rng.choice(["gesv", "gesv", "gesv", "getrf", "getrf_f32", "factor_solve_f32", "getrs", "vbatched", "adjoint",
                     "iteref_batched", "dense", "dense_iteref"])
    if op in ("gesv", "factor_solve_f32", "getrs"):
        n = _log(rng, 4, 512)
        c = {"op": op, "batch": _batch_for(rng, n, 10 ** 8), "n": n, "ld": n + rng.choice([0, 0, 0, 1, 4, 13]),
             "nrhs": _log(rng, 1, 16)}
        if op == "getrs":
            c["trans"] = rng.random() < 0.5
        return c
    if op in ("getrf", "getrf_f32"):
        m, n = _log(rng, 8, 700), _log(rng, 8, 700)
        if rng.random() < 0.5:
            n = m
        return {"op": op, "batch": _batch_for(rng, max(m, n), 5 * 10 ** 7), "m": m, "n": n,
                "ld": m + rng.choice([0, 0, 0, 1, 4, 13])}
    if op == "vbatched":
        nmin = _log(rng, 2, 128)
        nmax = _log(rng, nmin + 1, 512)
        return {"op": op, "batch": _log(rng, 20, 6000), "nmin": nmin, "nmax": nmax, "rmax": rng.randint(1, 16)}
    if op == "adjoint":
        n = _log(rng, 4, 256)
        return {"op": op, "dtype": rng.choice(["f64", "f32"]), "batch": _batch_for(rng, n, 5 * 10 ** 7), "n": n,
                "nrhs": _log(rng, 1, 16)}
    if op == "iteref_batched":
        n = _log(rng, 32, 512)
        return {"op": op, "batch": _batch_for(rng, n, 10 ** 8), "n": n, "ld": n + rng.choice([0, 0, 1]),
                "nrhs": _log(rng, 1, 4), "facto": rng.choice(["fp16", "bf16x3", "fp32"]),
                "solver": rng.choice(["ir", "gmres"])}
    if op == "dense":
        return {"op": op, "n": _log(rng, 400, 12000), "nrhs": rng.choice([1, 1, 4])}
    return {"op": op, "n": _log(rng, 700, 16000), "nrhs": 1, "facto": rng.choice(["fp16", "bf16x3"]),
            "solver": rng.choice(["ir", "gmres"])}


# --------------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(shape, dtype, g):
    return torch.empty(shape, dtype=dtype, device="cuda").uniform_(-1.0, 1.0, generator=g)


def _matrices(batch, m, n, ld, dtype, g):
    """(batch, n, ld): rows m .. ld-1 are padding."""
    A = _uniform((batch, n, ld), dtype, g)
    k = min(m, n)
    # column j of each matrix, j < k, gets its larger entry in a row of its own
    rows = torch.argsort(torch.rand((batch, m), device="cuda", generator=g), dim=1)[:, :k, None]
    A[:, :k].scatter_add_(2, rows, torch.full(rows.shape, math.sqrt(n), dtype=dtype, device="cuda"))
    return A


def _one_matrix(n, g):
    A = _uniform((n, n), torch.float64, g)
    rows = torch.randperm(n, device="cuda", generator=g)
    A[torch.arange(n, device="cuda"), rows] += math.sqrt(n)
    return A


def _vbatch_sizes(case):
    """The orders and right-hand side counts: part of the case, the same for every seed."""
    r = np.random.default_rng([case["batch"], case["nmin"], case["nmax"], case["rmax"]])
    ns = r.integers(case["nmin"], case["nmax"] + 1, case["batch"]).astype(np.int32)
    rs = r.integers(1, case["rmax"] + 1, case["batch"]).astype(np.int32)
    return ns, rs


def _vbatch_data(ns, rs, seed):
    """The packed matrices and right-hand sides (one more element at the end, as VBatch holds them)."""
    g = _generator(seed)
    size_a, size_b = int((ns.astype(np.int64) ** 2).sum()), int((ns.astype(np.int64) * rs).sum())
    A, B = _uniform(size_a + 1, torch.float64, g), _uniform(size_b + 1, torch.float64, g)
    offs = np.concatenate([[0], np.cumsum(ns.astype(np.int64) ** 2)[:-1]])
    r = np.random.default_rng(seed + 1)
    at = np.concatenate([o + np.arange(n) * n + r.permutation(n) for o, n in zip(offs, ns.astype(np.int64))])
    big = np.repeat(np.sqrt(ns.astype(np.float64)), ns)
    A[torch.from_numpy(at).cuda()] += torch.from_numpy(big).cuda()
    return A, B


def _inputs(case, seed):
    """The call's input tensors, from the seed alone."""
    g, op = _generator(seed), case["op"]
    if op in ("gesv", "getrs", "iteref_batched"):
        b, n, ld = case["batch"], case["n"], case["ld"]
        return _matrices(b, n, n, ld, torch.float64, g), _uniform((b, case["nrhs"], ld), torch.float64, g)
    if op == "factor_solve_f32":
        b, n, ld = case["batch"], case["n"], case["ld"]
        return _matrices(b, n, n, ld, torch.float32, g), _uniform((b, case["nrhs"], ld), torch.float32, g)
    if op in ("getrf", "getrf_f32"):
        return (_matrices(case["batch"], case["m"], case["n"], case["ld"],
                          torch.float64 if op == "getrf" else torch.float32, g),)
    if op == "adjoint":
        b, n, r, dt = case["batch"], case["n"], case["nrhs"], DTYPES[case["dtype"]]
        A = _matrices(b, n, n, n, dt, g)
        return A, _uniform((b, n, r), dt, g), _uniform((b, n, r), dt, g)
    if op in ("dense", "dense_iteref"):
        n = case["n"]
        return _one_matrix(n, g), _uniform((case["nrhs"], n), torch.float64, g)
    raise ValueError(op)


def prepare(case, seed):
    op = case["op"]
    if op == "vbatched":
        ns, rs = _vbatch_sizes(case)
        A0, B0 = _vbatch_data(ns, rs, seed)
        A, B = mb.VBatch(ns, ns), mb.VBatch(ns, rs)
        A.data.copy_(A0)
        B.data.copy_(B0)
        ipiv = mb.IpivV(ns)
        info = torch.zeros(len(ns), dtype=torch.int32, device="cuda")
        plan = mb.VbatchedPlan(ns, rs, variants=autotune.load_variants(ns, rs))
        plan.capture(A, B, ipiv, info)
        return {"op": op, "A0": A0, "B0": B0, "A": A, "B": B, "ipiv": ipiv, "info": info, "plan": plan}
    ins = _inputs(case, seed)
    s = {"op": op, "ins": ins, "case": dict(case)}
    if op == "getrs":
        s["ipiv"], s["info"] = mb.dgetrf_batched(ins[0], m=case["n"])
        s["B"] = torch.empty_like(ins[1])
    elif op == "adjoint":
        s["A"], s["B"] = ins[0].requires_grad_(), ins[1].requires_grad_()
    elif op in ("gesv", "factor_solve_f32", "dense"):
        s["A"], s["B"] = torch.empty_like(ins[0]), torch.empty_like(ins[1])
    elif op in ("getrf", "getrf_f32"):
        s["A"] = torch.empty_like(ins[0])
    elif op == "iteref_batched":
        s["X"] = torch.zeros_like(ins[1])
    return s


# --------------------------------------------------------------------------- one pass
def run(s):
    op = s["op"]
    if op == "vbatched":
        s["A"].data.copy_(s["A0"])
        s["B"].data.copy_(s["B0"])
        s["plan"].replay()
        return {"LU": s["A"].data, "X": s["B"].data, "ipiv": s["ipiv"].data, "info": s["info"]}
    ins, case = s["ins"], s["case"]
    if op == "gesv":
        A, B = s["A"].copy_(ins[0]), s["B"].copy_(ins[1])
        ipiv, info = mb.dgesv_batched(A, B)
        return {"LU": A, "X": B, "ipiv": ipiv, "info": info}
    if op == "getrf":
        A = s["A"].copy_(ins[0])
        ipiv, info = mb.dgetrf_batched(A, m=case["m"])
        return {"LU": A, "ipiv": ipiv, "info": info}
    if op == "getrf_f32":
        A = s["A"].copy_(ins[0])
        ipiv, info = mb.sgetrf_batched(A, m=case["m"])
        return {"LU": A, "ipiv": ipiv, "info": info}
    if op == "factor_solve_f32":
        A, B = s["A"].copy_(ins[0]), s["B"].copy_(ins[1])
        ipiv, info = mb.sgetrf_batched(A, m=case["n"])
        mb.sgetrs_batched(MagmaNoTrans, A, ipiv, B)
        return {"LU": A, "X": B, "ipiv": ipiv, "info": info}
    if op == "getrs":
        B = s["B"].copy_(ins[1])
        mb.dgetrs_batched(MagmaTrans if case["trans"] else MagmaNoTrans, ins[0], s["ipiv"], B)
        return {"X": B}
    if op == "adjoint":
        X = solve(s["A"], s["B"])
        gA, gB = torch.autograd.grad(X, (s["A"], s["B"]), ins[2])
        return {"X": X, "gA": gA, "gB": gB}
    if op == "iteref_batched":
        # the sweep counts are left out: they say how the solver got there
        X, _, info = iteref.dxgesv_iteref_batched(ins[0], ins[1], X=s["X"], facto=case["facto"],
                                                 solver=case["solver"])
        return {"X": X, "info": info}
    if op == "dense":
        A, B = s["A"].copy_(ins[0]), s["B"].copy_(ins[1])
        ipiv, info = dense.getrf_gpu(A)
        dense.getrs_gpu(A, ipiv, B)
        return {"LU": A, "X": B, "ipiv": ipiv, "info": info}
    X, _, _, _, info = iteref.dhgesv_iteref_gpu(ins[0], ins[1], facto=case["facto"], solver=case["solver"])
    return {"X": X, "info": info}


# --------------------------------------------------------------------------- what a pass cannot do without
def _getrf_flops(n):
    return 2 * n ** 3 / 3 - n * n / 2 + 5 * n / 6


def _gesv_work(n, r, elem):
    """One system: A and B read, LU, X, ipiv and info written."""
    return 2 * elem * n * (n + r) + 4 * n + 4, _getrf_flops(n) + r * (2 * n * n - n)


def work(case):
    op = case["op"]
    if op == "vbatched":
        ns, rs = _vbatch_sizes(case)
        w = [_gesv_work(float(n), float(r), 8) for n, r in zip(ns, rs)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    if op in ("gesv", "factor_solve_f32"):
        b, f = _gesv_work(case["n"], case["nrhs"], 4 if op.endswith("f32") else 8)
        return {"bytes": case["batch"] * b, "flops": case["batch"] * f}
    if op in ("getrf", "getrf_f32"):
        m, n, e = case["m"], case["n"], 4 if op.endswith("f32") else 8
        f = sum(2.0 * (m - k - 1) * (n - k - 1) + (m - k - 1) for k in range(min(m, n)))
        return {"bytes": case["batch"] * (2 * e * m * n + 4 * min(m, n) + 4), "flops": case["batch"] * f}
    if op == "getrs":
        n, r = case["n"], case["nrhs"]
        return {"bytes": case["batch"] * (8 * n * n + 16 * n * r + 4 * n), "flops": case["batch"] * r * (2 * n * n - n)}
    if op == "adjoint":
        # forward: A, B read, X written (the factors and pivots are kept for the backward pass: written, then read);
        # backward: G and X read, gA and gB written
        n, r, e = case["n"], case["nrhs"], 8 if case["dtype"] == "f64" else 4
        return {"bytes": case["batch"] * (e * (4 * n * n + 5 * n * r) + 8 * n + 4),
                "flops": case["batch"] * (_getrf_flops(n) + 2 * r * (2 * n * n - n) + 2 * n * n * r)}
    n, r = case["n"], case["nrhs"]
    f = _getrf_flops(n) + r * (2 * n * n - n)
    if op == "iteref_batched":
        return {"bytes": case["batch"] * (8 * n * n + 16 * n * r + 4), "flops": case["batch"] * f}
    if op == "dense":
        return {"bytes": 16 * n * n + 16 * n * r + 4 * n, "flops": f}
    return {"bytes": 8 * n * n + 16 * n * r, "flops": f}


# --------------------------------------------------------------------------- the same in 64 bits, from torch on the host
def _factor(M):
    """Column-major (..., n, m) -> the factors in the same layout."""
    return torch.linalg.lu_factor(M.double().cpu().transpose(-1, -2))[0].transpose(-1, -2)


def _solved(M, B, trans=False):
    """Column-major M (..., n, n) and B (..., r, n) -> X (..., r, n)."""
    M, B = M.double().cpu(), B.double().cpu()
    return torch.linalg.solve(M if trans else M.transpose(-1, -2), B.transpose(-1, -2)).transpose(-1, -2)


def _with_padding(F, M):
    """The factors F (m rows) with the padding rows that M came with."""
    out = M.double().cpu().clone()
    out[..., : F.shape[-1]] = F
    return out


def exact(case, seed):
    op = case["op"]
    if op == "vbatched":
        ns, rs = _vbatch_sizes(case)
        A, B = (t.cpu() for t in _vbatch_data(ns, rs, seed))
        oa = np.concatenate([[0], np.cumsum(ns.astype(np.int64) ** 2)])
        ob = np.concatenate([[0], np.cumsum(ns.astype(np.int64) * rs)])
        for i, (n, r) in enumerate(zip(ns.tolist(), rs.tolist())):
            M, Y = A[oa[i]:oa[i + 1]].view(n, n), B[ob[i]:ob[i + 1]].view(r, n)
            LU, p = torch.linalg.lu_factor(M.T)
            Y.copy_(torch.linalg.lu_solve(LU, p, Y.T).T)
            M.copy_(LU.T)
        return {"LU": A, "X": B, "ipiv": None, "info": None}
    if case["n"] > 12000:
        return None
    ins = _inputs(case, seed)
    if op in ("getrf", "getrf_f32"):
        return {"LU": _with_padding(_factor(ins[0][..., : case["m"]]), ins[0]), "ipiv": None, "info": None}
    if op == "adjoint":
        A, B, G = (t.double().cpu() for t in ins)
        X, gB = torch.linalg.solve(A, B), torch.linalg.solve(A.transpose(1, 2), G)
        return {"X": X, "gA": -torch.matmul(gB, X.transpose(1, 2).contiguous()), "gB": gB}
    n = case["n"]
    M, B = ins[0][..., :n], ins[1][..., :n]
    if op in ("dense_iteref", "iteref_batched"):
        return {"X": _with_padding(_solved(M, B), torch.zeros_like(ins[1])), "info": None}
    X = _with_padding(_solved(M, B, op == "getrs" and case["trans"]), ins[1])
    return {"X": X} if op == "getrs" else {"LU": _with_padding(_factor(M), ins[0]), "X": X, "ipiv": None, "info": None}
