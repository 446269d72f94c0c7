"""The work that programs have this library do, as cases that can be timed.

A case is one product through the public entry points, with the matrix handle
optimized beforehand and the vectors or dense operands resident in HBM, as an
iterative solver, an eigensolver or a graph network calls it in its inner loop:

  kind "spmv"   y = alpha op(A) x + beta y, CSR or BSR handle after optimize()
  kind "spmm"   C = alpha A B + beta C, k columns, row-major B and C
  kind "batch"  Y_p = A_p X_p of many small matrices in one launch

Matrices come from the five families the library's selector knows (2-D / 3-D
stencils, banded, power-law, uniform random rows, dense 4 x 4 / 8 x 8 blocks on
a 3-D block grid); values and operands are drawn from the seed.  `prec` is the
arithmetic of the product: "f64", "f32", or "bf16" (a single-precision handle
whose values are stored in BF16).
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "perf-libs-sparse_amd"))

import plsparse as P  # noqa: E402
from plsparse import workloads as W  # noqa: E402


def listed():
    return [
        # The smallest matrix anybody iterates with: the inner loop of a 2-D
        # Poisson solver.  Everything is cache-resident; launch and call latency.
        {"name": "spmv_laplace5_f64", "kind": "spmv", "matrix": "laplace5", "grid": 316,
         "prec": "f64", "alpha": 1.0, "beta": 0.5},
        # The ordinary solver product: a 27-point operator of a 3-D grid.
        {"name": "spmv_stencil27_f64", "kind": "spmv", "matrix": "stencil27", "grid": 96,
         "prec": "f64", "alpha": 1.0, "beta": 0.0},
        # The headline product: PageRank-like iteration over a 4M-vertex graph,
        # uneven rows, scattered columns.
        {"name": "spmv_powerlaw_f64", "kind": "spmv", "matrix": "powerlaw", "rows": 4194304,
         "prec": "f64", "alpha": 1.0, "beta": 0.0},
        # The same kind of graph, odd size, with weights stored in BF16 and damping.
        {"name": "spmv_powerlaw_bf16", "kind": "spmv", "matrix": "powerlaw", "rows": 1000003,
         "prec": "bf16", "alpha": 0.85, "beta": 0.15},
        # The adjoint product of a bidiagonalisation: banded rows, op = TRANS.
        {"name": "spmv_banded_f32_trans", "kind": "spmv", "matrix": "banded", "rows": 700001,
         "band": 256, "lo": 5, "hi": 40, "prec": "f32", "alpha": 1.0, "beta": 0.0, "trans": True},
        # A vector-valued finite-element operator: 4 unknowns per grid point.
        {"name": "spmv_bsr4_f64", "kind": "spmv", "matrix": "blocks", "grid": 48, "b": 4,
         "prec": "f64", "alpha": 1.0, "beta": 0.0},
        # A few right-hand sides at once (block Krylov), single precision.
        {"name": "spmm_stencil27_f32_k8", "kind": "spmm", "matrix": "stencil27", "grid": 80, "k": 8,
         "prec": "f32", "alpha": 1.0, "beta": 0.0},
        # A block eigensolver's basis.
        {"name": "spmm_stencil27_f64_k32", "kind": "spmm", "matrix": "stencil27", "grid": 96, "k": 32,
         "prec": "f64", "alpha": 1.0, "beta": 0.0},
        # Many right-hand sides: the widest B the benchmark multiplies by.
        {"name": "spmm_stencil27_f64_k128", "kind": "spmm", "matrix": "stencil27", "grid": 80, "k": 128,
         "prec": "f64", "alpha": 1.0, "beta": 0.0},
        # Neighbour aggregation of a graph network: scattered rows of a feature matrix.
        {"name": "spmm_powerlaw_f32_k64", "kind": "spmm", "matrix": "powerlaw", "rows": 262144, "k": 64,
         "prec": "f32", "alpha": 1.0, "beta": 0.0},
        # Block rows times a block basis, 8 unknowns per grid point.
        {"name": "spmm_bsr8_f64_k32", "kind": "spmm", "matrix": "blocks", "grid": 32, "b": 8, "k": 32,
         "prec": "f64", "alpha": 1.0, "beta": 0.0},
        # Many independent uneven problems, 1, 4 or 16 right-hand sides each.
        {"name": "batch_banded_f64", "kind": "batch", "problems": 256, "prec": "f64",
         "alpha": 1.0, "beta": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Sizes over the listed ranges: 3,000 to 1M rows, 5 to 60 non-zeros per
    row, 1 to 128 columns of B, every family, precision, op and beta."""
    kind = rng.choice(["spmv", "spmv", "spmm", "spmm", "spmm", "batch"])
    c = {"kind": kind, "prec": rng.choice(["f64", "f64", "f32", "bf16"]),
         "alpha": rng.choice([1.0, 1.0, -1.0, 0.85]), "beta": rng.choice([0.0, 0.0, 1.0, 0.5])}
    if kind == "batch":
        c["problems"] = _log(rng, 16, 256)
        return c
    if kind == "spmm":
        c["k"] = rng.choice([_log(rng, 1, 128), rng.choice([4, 8, 16, 32, 64, 128])])
    # at most about 20M non-zeros for SpMV, 150M non-zero columns for SpMM
    cap = 1.0 if kind == "spmv" else min(1.0, 8.0 / c["k"])
    m = c["matrix"] = rng.choice(["laplace5", "stencil27", "powerlaw", "banded", "uniform", "blocks"])
    if m == "laplace5":
        c["grid"] = _log(rng, 60, 1000 * math.sqrt(cap))
    elif m == "stencil27":
        c["grid"] = _log(rng, 15, 90 * cap ** (1 / 3))
    elif m == "powerlaw":
        c["rows"] = _log(rng, 3000, 1000000 * cap)
    elif m == "blocks":
        c["b"] = rng.choice([4, 8])
        c["grid"] = _log(rng, 6, (44 if c["b"] == 4 else 28) * cap ** (1 / 3))
    else:
        c["lo"] = rng.randint(1, 12)
        c["hi"] = c["lo"] + rng.randint(0, 48)
        c["rows"] = _log(rng, 3000, 600000 * cap)
        if m == "banded":
            c["band"] = rng.randint(64, 600)
    if kind == "spmv" and m != "blocks" and rng.random() < 0.25:
        c["trans"] = True
    return c


def _csr(case, seed):
    """(row_ptr, col, vals as float64) of a square CSR matrix."""
    m = case["matrix"]
    if m == "laplace5":
        rp, ci, v = W.laplace2d(case["grid"])
    elif m == "stencil27":
        rp, ci, v = W.stencil27(case["grid"])
    elif m == "powerlaw":
        return W.powerlaw(case["rows"], seed)
    elif m == "banded":
        return W.banded(case["rows"], case["band"], case["lo"], case["hi"], seed)
    else:
        return W.random_rows(case["rows"], case["rows"], case["lo"], case["hi"], seed)
    return rp, ci, v * W.uniform(len(v), seed, 0.5, 1.5)  # a variable coefficient


def _tdtype(case):
    return torch.float64 if case["prec"] == "f64" else torch.float32


def _operands(case, rows, cols, seed):
    """Uniform [-1, 1] operand (x or B) and the old content of the result (y or C)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = case.get("k", 1)
    shape = (cols, k) if case["kind"] == "spmm" else (cols,)
    out = (rows, k) if case["kind"] == "spmm" else (rows,)
    x = torch.rand(shape, generator=g, dtype=_tdtype(case), device="cuda") * 2 - 1
    y = torch.rand(out, generator=g, dtype=_tdtype(case), device="cuda") * 2 - 1
    return x, y


def _sizes(case):
    """(rows, bandwidth, right-hand sides) of each problem of a batch: rows
    log-uniform in [256, 65536], bandwidth 32 to 512, 1, 4 or 16 columns."""
    rng = np.random.default_rng(case["problems"])
    return [(int(round(256 * 256 ** rng.random())), int(rng.integers(32, 513)),
             int(rng.choice([1, 4, 16]))) for _ in range(case["problems"])]


def _problems(case, seed):
    probs = [(m, *W.banded(m, w, 5, 40, seed * 1000003 + p), k)  # 5 to 40 non-zeros per row
             for p, (m, w, k) in enumerate(_sizes(case))]
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = sum(p[0] * p[4] for p in probs)
    x = torch.rand(n, generator=g, dtype=_tdtype(case), device="cuda") * 2 - 1
    y = torch.rand(n, generator=g, dtype=_tdtype(case), device="cuda") * 2 - 1
    at = np.cumsum([0] + [p[0] * p[4] for p in probs])
    return probs, x, y, at


def prepare(case, seed):
    P.set_stream(torch.cuda.current_stream().cuda_stream)
    hdt = np.float64 if case["prec"] == "f64" else np.float32
    if case["kind"] == "batch":
        probs, x, y, at = _problems(case, seed)
        mats = [P.SpMat.csr(m, m, rp, ci, v.astype(hdt, copy=False), flags=P.CREATE_NOCOPY)
                for (m, rp, ci, v, _) in probs]
        b = P.Batch(mats, [p[4] for p in probs],
                    P.VALUES_BF16 if case["prec"] == "bf16" else P.VALUES_NATIVE)
        es = x.element_size()
        b.set_operands([x.data_ptr() + es * int(a) for a in at[:-1]],
                       [y.data_ptr() + es * int(a) for a in at[:-1]])
        b.optimize(autotune=True)
        return {"case": case, "batch": b, "x": x, "y": y}
    if case["matrix"] == "blocks":
        g, b = case["grid"], case["b"]
        rp, ci, v = W.block_stencil(g, g, g, b, seed)
        m = g * g * g * b
        A = P.SpMat.bsr(P.ROW_MAJOR, m, m, b, rp, ci, v.astype(hdt, copy=False), flags=P.CREATE_NOCOPY)
    else:
        rp, ci, v = _csr(case, seed)
        m = len(rp) - 1
        A = P.SpMat.csr(m, m, rp, ci, v.astype(hdt, copy=False), flags=P.CREATE_NOCOPY)
    if case["prec"] == "bf16":
        A.set_precision(P.VALUES_BF16)
    x, y = _operands(case, m, m, seed)
    op = P.TRANS if case.get("trans") else P.NOTRANS
    if case["kind"] == "spmv":
        A.hint(P.HINT_SPMV_OPERATION, op)
        A.hint(P.HINT_SPMV_INVOCATIONS, P.INVOCATIONS_MANY)
        A.optimize()
    else:  # the first product builds the handle's SpMM plan
        k, c = case["k"], torch.empty_like(y)
        A.spmm_async(k, x.data_ptr(), k, c.data_ptr(), k)
        torch.cuda.synchronize()
    return {"case": case, "A": A, "x": x, "y": y, "op": op}


def run(state):
    c, y = state["case"], state["y"]
    if c["kind"] == "batch":
        state["batch"].exec(c["alpha"], c["beta"])
    elif c["kind"] == "spmv":
        state["A"].spmv_async(state["x"].data_ptr(), y.data_ptr(), c["alpha"], c["beta"], state["op"])
    else:
        k = c["k"]
        state["A"].spmm_async(k, state["x"].data_ptr(), k, y.data_ptr(), k, c["alpha"], c["beta"])
    return y


def _product(case, rp, ci, v, x, y, trans=False):
    """alpha op(A) x + beta y in float64 (x, y: one row per row of op(A)), by
    gathering and adding on the GPU a slice of the non-zeros at a time."""
    rp = torch.from_numpy(np.asarray(rp, np.int64)).cuda()
    ci = torch.from_numpy(np.asarray(ci, np.int64)).cuda()
    v = torch.from_numpy(np.asarray(v, np.float64)).cuda()
    if case["prec"] != "f64":
        v = v.float().to(torch.bfloat16).double() if case["prec"] == "bf16" else v.float().double()
    row = torch.repeat_interleave(torch.arange(len(rp) - 1, device="cuda"), rp[1:] - rp[:-1])
    if trans:
        row, ci = ci, row
    x2 = x.double().reshape(x.shape[0], -1)
    out = torch.zeros((y.shape[0], x2.shape[1]), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // x2.shape[1])
    for a in range(0, len(v), step):
        s = slice(a, a + step)
        out.index_add_(0, row[s], v[s, None] * x2[ci[s]])
    return (case["alpha"] * out).reshape(y.shape) + case["beta"] * y.double()


def exact(case, seed):
    if case["kind"] == "batch":
        probs, x, y, at = _problems(case, seed)
        out = torch.empty_like(y, dtype=torch.float64)
        for (m, rp, ci, v, k), a in zip(probs, at):
            s = slice(int(a), int(a) + m * k)
            out[s] = _product(case, rp, ci, v, x[s].view(m, k), y[s].view(m, k)).reshape(-1)
        return out
    if case["matrix"] == "blocks":
        g, b = case["grid"], case["b"]
        rp, ci, v = W.block_stencil(g, g, g, b, seed)
        # every stored value as an entry: block row * b + i, block column * b + j
        row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
        row = row[:, None, None] * b + np.arange(b)[None, :, None] + np.zeros((1, 1, b), np.int64)
        col = ci.astype(np.int64)[:, None, None] * b + np.zeros((1, b, 1), np.int64) + np.arange(b)[None, None, :]
        order = np.argsort(row.reshape(-1), kind="stable")
        ci, v = col.reshape(-1)[order], v[order]
        rp = np.concatenate([[0], np.cumsum(np.repeat(np.diff(rp) * b, b))])
    else:
        rp, ci, v = _csr(case, seed)
    m = len(rp) - 1
    x, y = _operands(case, m, m, seed)
    return _product(case, rp, ci, v, x, y, case.get("trans", False))


def work(case):
    """Each stored value and index once, the operand once, the result once
    (twice when it is also read), and two operations per product."""
    sv, sx = {"f64": (8, 8), "f32": (4, 4), "bf16": (2, 4)}[case["prec"]]
    rw = 2 if case["beta"] != 0.0 else 1
    if case["kind"] == "batch":
        s = _sizes(case)
        rows, vec = sum(m for m, _, _ in s), sum(m * k for m, _, k in s)
        return {"bytes": 22.5 * rows * (sv + 4) + rows * 4 + vec * sx * (1 + rw), "flops": 2 * 22.5 * vec}
    k, m = case.get("k", 1), case["matrix"]
    if m == "blocks":
        g, b = case["grid"], case["b"]
        nb = (3 * g - 2) ** 3
        n, nnz = g ** 3 * b, nb * b * b
        stored = nnz * sv + nb * 4 + (g ** 3 + 1) * 4
    else:
        if m == "laplace5":
            n, nnz = case["grid"] ** 2, 5 * case["grid"] ** 2 - 4 * case["grid"]
        elif m == "stencil27":
            n, nnz = case["grid"] ** 3, (3 * case["grid"] - 2) ** 3
        elif m == "powerlaw":
            n, nnz = case["rows"], 20.1 * case["rows"]
        else:
            n, nnz = case["rows"], (case["lo"] + case["hi"]) / 2 * case["rows"]
        stored = nnz * (sv + 4) + (n + 1) * 4
    return {"bytes": stored + n * k * sx * (1 + rw), "flops": 2 * nnz * k}
