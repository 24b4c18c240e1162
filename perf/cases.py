"""Workloads of the CSR sparse x dense path, for timing and comparing builds.

Each case is one pass through the package's public entry points on matrices
of the benchmark's and the tests' families (2D Laplacian, 3D Poisson, random
rows, power-law rows, banded), made on the GPU from a seed alone:

- ``spmv``: ``A @ x``;
- ``spmm``: ``A @ X`` with k columns;
- ``batch``: ``csr_batched_matvec`` over ``batch`` vectors;
- ``adjoint``: ``csr_matvec_transpose`` (k = 0) or ``csr_matmul_transpose``;
- ``train``: one step of a loop that writes new values into the matrix
  (``trained``) or keeps them: the product, and its gradients in the values
  (``trained``) and in the dense operand;
- ``solve``: ``linalg.cg / bicgstab / minres / gmres`` on the shifted
  operator of an implicit time step (diffusion; ``convection`` makes it
  non-symmetric), to a relative residual of 1e-5 from zero.

``listed`` gives the fixed cases, ``draw`` one more of the same ranges.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "mlx-sparse_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mlx_sparse as ms  # noqa: E402
from mlx_sparse import linalg  # noqa: E402

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16,
           "c64": torch.complex64}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "c64": 8}
_INDEX = {"i32": torch.int32, "i64": torch.int64}


def _case(op, matrix, n, *, dtype="f32", index="i32", per_row=16, cols=0, k=0, batch=0,
          trained=False, solver="", convection=0.0, name=None):
    """``n``: rows (grid side for the stencils); ``per_row``: values per row
    (random) or half bandwidth (banded); ``cols``: columns, 0 for square."""
    case = {"op": op, "matrix": matrix, "n": n, "dtype": dtype, "index": index,
            "per_row": per_row, "cols": cols, "k": k, "batch": batch, "trained": trained,
            "solver": solver, "convection": convection}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest call: one product with a 2,209-row operator, as a host loop
        # (a time step, a hand-written solver) makes it thousands of times; launch bound
        _case("spmv", "laplacian", 47, name="spmv_small"),
        # the benchmark's headline: scattered columns over an x far above any cache
        _case("spmv", "random", 4_194_304, name="spmv_random"),
        # a web-like graph: row lengths from 1 to 187,500, 64-bit indices, odd size
        _case("spmv", "powerlaw", 1_500_007, index="i64", name="spmv_powerlaw"),
        # a banded operator kept in 16 bits, odd size
        _case("spmv", "banded", 786_433, dtype="bf16", per_row=32, name="spmv_banded_bf16"),
        # a block of 64 vectors through the 3D stencil (block methods, fields)
        _case("spmm", "poisson", 128, k=64, name="spmm_poisson"),
        # neighbour aggregation of 16-bit features on a graph, ragged feature width
        _case("spmm", "random", 300_007, dtype="f16", per_row=20, k=100, name="spmm_graph_f16"),
        # a handful of complex vectors at once (several sources of one wave problem)
        _case("batch", "banded", 200_003, dtype="c64", per_row=8, batch=6, name="batch_c64"),
        # A^T x without a stored transpose (normal equations, one-off adjoints), rectangular
        _case("adjoint", "random", 1_000_003, per_row=12, cols=600_011, name="adjoint_random"),
        # a learned linear operator: new values each step, gradients of values and x
        _case("train", "random", 1_300_021, per_row=16, trained=True, name="train_spmv"),
        # graph attention on a web-like graph: new edge weights each step, gradients of the
        # weights and of the node features
        _case("train", "powerlaw", 300_007, k=32, trained=True, name="train_spmm"),
        # a small implicit step solved with conjugate gradients; latency bound
        _case("solve", "laplacian", 63, solver="cg", name="solve_cg_small"),
        # a large non-symmetric implicit step
        _case("solve", "poisson", 96, solver="bicgstab", convection=0.3, name="solve_bicgstab"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["spmv"] * 3 + ["spmm"] * 2 + ["train"] * 2 + ["solve"] * 2
                    + ["batch", "adjoint"])
    if op == "solve":
        solver = rng.choice(["cg", "bicgstab", "minres", "gmres"])
        convection = rng.uniform(0.1, 0.4) if solver in ("bicgstab", "gmres") else 0.0
        matrix = rng.choice(["laplacian", "poisson"])
        n = _log(rng, 30, 700) if matrix == "laplacian" else _log(rng, 10, 80)
        return _case(op, matrix, n, index=rng.choice(["i32", "i32", "i64"]), solver=solver,
                     convection=round(convection, 3))
    matrix = rng.choice(["laplacian", "poisson", "random", "random", "powerlaw", "banded"])
    if op == "train":
        dtype = rng.choice(["f32", "f32", "bf16"])
    else:
        dtype = rng.choice(["f32", "f32", "f32", "f16", "bf16", "c64"])
    index = rng.choice(["i32", "i32", "i64"])
    k = batch = 0
    if op == "spmm" or (op in ("train", "adjoint") and rng.random() < 0.5):
        k = rng.choice([4, 8, 16, 32, 64, 128, _log(rng, 2, 200), _log(rng, 2, 200)])
    if op == "batch":
        batch = _log(rng, 2, 48)
    width = max(k, batch, 1) * (2 if dtype == "c64" else 1)
    per_row, cols = 16, 0
    mean = {"laplacian": 5, "poisson": 7, "powerlaw": 12}.get(matrix)
    if matrix == "random":
        mean = per_row = _log(rng, 3, 40)
    elif matrix == "banded":
        per_row = _log(rng, 2, 48)
        mean = 1 + 1.3 * per_row
    # the work of the largest listed ones: 40 M values, 5e8 products, 8e7 dense values
    most = min(4_000_000, 4e7 / mean, 5e8 / (mean * width), 8e7 / width)
    if matrix == "powerlaw" and width > 1:
        most = min(most, 300_000)
    n = _log(rng, 1_500, max(3_000, most))
    if matrix == "laplacian":
        n = max(30, round(n ** 0.5))
    elif matrix == "poisson":
        n = max(11, round(n ** (1 / 3)))
    elif matrix == "random" and rng.random() < 0.4:
        cols = max(1_000, int(n * rng.uniform(0.3, 2.0)))
    return _case(op, matrix, n, dtype=dtype, index=index, per_row=per_row, cols=cols, k=k,
                 batch=batch, trained=op == "train" and rng.random() < 0.6)


# -- the matrices, on the GPU ----------------------------------------------
def _offsets(case):
    """(row count, [(column offset, axis, step, value)]) of a stencil, by
    increasing column; the diagonal has axis -1."""
    g, dims = case["n"], (2 if case["matrix"] == "laplacian" else 3)
    shift = 0.5 if case["op"] == "solve" else 0.0
    c = case["convection"]
    low = [(-(g ** a), a, -1, -1.0 - c) for a in range(dims - 1, -1, -1)]
    high = [(g ** a, a, 1, -1.0 + c) for a in range(dims)]
    return g ** dims, low + [(0, -1, 0, 2.0 * dims + shift)] + high


def _counts(case):
    """(rows, columns, stored values) of a case's matrix; the values of
    ``banded`` and ``powerlaw`` to a fraction of a percent."""
    if case["matrix"] in ("laplacian", "poisson"):
        rows, offs = _offsets(case)
        return rows, rows, rows * len(offs) - (len(offs) - 1) * (rows // case["n"])
    n = case["n"]
    cols = case["cols"] or n
    if case["matrix"] == "random":
        return n, cols, n * case["per_row"]
    if case["matrix"] == "banded":
        return n, n, n * (1 + 13 * case["per_row"] // 10)
    cap = min(200_000, max(1, n // 8))
    return n, n, int(n * (math.log(cap) + 0.577))


def _stencil(case, dev):
    rows, offs = _offsets(case)
    g = case["n"]
    idx = torch.arange(rows, device=dev)
    cols, keep = [], []
    for off, axis, step, _ in offs:
        cols.append(idx + off)
        if axis < 0:
            keep.append(torch.ones(rows, dtype=torch.bool, device=dev))
        else:
            at = idx // g ** axis % g + step
            keep.append((at >= 0) & (at < g))
    cols, keep = torch.stack(cols, 1), torch.stack(keep, 1)
    vals = torch.tensor([o[3] for o in offs], device=dev).expand(rows, -1)
    return keep.sum(1), cols[keep], vals[keep].contiguous(), rows


def _normal(gen, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device=gen.device, dtype=dtype)


def _random(case, gen):
    rows, cols, per = case["n"], case["cols"] or case["n"], case["per_row"]
    dev = gen.device
    c = torch.randint(cols, (rows, per), generator=gen, device=dev, dtype=torch.int32)
    c = c.sort(dim=1).values
    while True:  # rows with a repeated column are drawn again
        bad = (c[:, 1:] == c[:, :-1]).any(1).nonzero()[:, 0]
        if bad.numel() == 0:
            break
        c[bad] = torch.randint(cols, (bad.numel(), per), generator=gen, device=dev,
                               dtype=torch.int32).sort(dim=1).values
    lengths = torch.full((rows,), per, device=dev)
    return lengths, c.reshape(-1), _normal(gen, rows * per), cols


def _power_law(case, gen):
    n, dev = case["n"], gen.device
    cap = min(200_000, max(1, n // 8))
    at = (torch.randperm(n, generator=gen, device=dev).double() + 0.5) / n
    lengths = (1.0 / at).long().clamp(max=cap)
    rows = torch.repeat_interleave(torch.arange(n, device=dev), lengths)
    key = rows * n + torch.randint(n, (rows.numel(),), generator=gen, device=dev)
    while True:  # a repeated column of a row is drawn again
        key = key.sort().values
        bad = (key[1:] == key[:-1]).nonzero()[:, 0]
        if bad.numel() == 0:
            break
        key[bad] = rows[bad] * n + torch.randint(n, (bad.numel(),), generator=gen, device=dev)
    return lengths, key % n, (1.0 / lengths[rows]).float(), n


def _banded(case, gen):
    n, hb, dev = case["n"], case["per_row"], gen.device
    offs = torch.arange(-hb, hb + 1, device=dev, dtype=torch.int32)
    cols = torch.arange(n, device=dev, dtype=torch.int32)[:, None] + offs
    valid = (cols >= 0) & (cols < n)
    # the diagonal and 65 % of the band, any of it
    order = torch.rand(n, 2 * hb + 1, generator=gen, device=dev)
    order[:, hb] = -1.0
    order = order.masked_fill_(~valid, 2.0).sort(dim=1, stable=True).indices
    keep = torch.zeros_like(valid).scatter_(1, order[:, :1 + 13 * hb // 10], True) & valid
    vals = _normal(gen, n, 2 * hb + 1)
    vals[:, hb] += 2.0 * hb + 6.0
    return keep.sum(1), cols[keep], vals[keep], n


def _inputs(case, seed):
    """(data, indices, indptr, shape, dense operands) of a case."""
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed) * 7919 + 17)
    dtype, index = _DTYPES[case["dtype"]], _INDEX[case["index"]]
    if case["matrix"] in ("laplacian", "poisson"):
        lengths, cols, vals, n_cols = _stencil(case, dev)
        if case["trained"]:
            vals = vals + 0.1 * _normal(gen, vals.numel())
    else:
        lengths, cols, vals, n_cols = {"random": _random, "powerlaw": _power_law,
                                       "banded": _banded}[case["matrix"]](case, gen)
    rows = lengths.numel()
    indptr = torch.zeros(rows + 1, dtype=torch.int64, device=dev)
    torch.cumsum(lengths, 0, out=indptr[1:])
    if dtype.is_complex:
        vals = torch.complex(vals, _normal(gen, vals.numel()))

    def dense(*shape):
        if dtype.is_complex:
            return _normal(gen, *shape, dtype=dtype)
        if len(shape) == 1:  # a field in [-1, 1]
            return (2.0 * torch.rand(*shape, generator=gen, device=dev) - 1.0).to(dtype)
        return _normal(gen, *shape).to(dtype)

    tail = (case["k"],) if case["k"] else ()
    op = case["op"]
    if op == "batch":
        operands = (dense(case["batch"], n_cols),)
    elif op == "adjoint":
        operands = (dense(rows, *tail),)
    elif op == "train":
        operands = (dense(n_cols, *tail), dense(rows, *tail))
    else:
        operands = (dense(n_cols, *tail),)
    return (vals.to(dtype), cols.to(index).contiguous(), indptr.to(index), (rows, n_cols),
            operands)


# -- one pass ----------------------------------------------------------------
def prepare(case, seed):
    data, indices, indptr, shape, operands = _inputs(case, seed)
    state = {"case": case, "operands": operands}
    if case["op"] == "train":
        if case["trained"]:
            state["values"] = data
            data = data.clone().requires_grad_(True)
        operands[0].requires_grad_(True)
    state["a"] = ms.csr_array((data, indices, indptr), shape=shape, sorted_indices=True)
    if case["op"] not in ("batch", "adjoint"):
        state["a"].plan()
    return state


def run(state):
    case, a, operands = state["case"], state["a"], state["operands"]
    op = case["op"]
    if op in ("spmv", "spmm"):
        return a @ operands[0]
    if op == "batch":
        return ms.csr_batched_matvec(a, operands[0])
    if op == "adjoint":
        if case["k"]:
            return ms.csr_matmul_transpose(a, operands[0])
        return ms.csr_matvec_transpose(a, operands[0])
    if op == "train":
        x, g = operands
        if case["trained"]:
            with torch.no_grad():
                a.data.copy_(state["values"])
        y = a @ x
        wanted = (a.data, x) if case["trained"] else (x,)
        return (y.detach(), *torch.autograd.grad(y, wanted, g))
    solver = getattr(linalg, case["solver"])
    x, info = solver(a, operands[0], rtol=1e-5)
    return x, info


def work(case):
    rows, cols, nnz = _counts(case)
    v, i = _BYTES[case["dtype"]], 4 if case["index"] == "i32" else 8
    width = max(case["k"], case["batch"], 1)
    mul = 8 if case["dtype"] == "c64" else 2
    matrix = nnz * (v + i) + (rows + 1) * i
    dense = (rows + cols) * width * v
    op = case["op"]
    if op == "train":
        # values, structure and both dense operands in; product and gradients out
        out = rows * width * v + cols * width * v + (nnz * v if case["trained"] else 0)
        new = nnz * v if case["trained"] else 0
        return {"bytes": matrix + new + dense + out,
                "flops": mul * nnz * width * (3 if case["trained"] else 2)}
    if op == "solve":
        # iterations to 1e-5 of these systems, measured; per iteration the
        # matrix for each product and the loop's vectors
        steps, products, vectors = {"cg": (24, 1, 11), "bicgstab": (21, 2, 20),
                                    "minres": (24, 2, 18), "gmres": (40, 1, 24)}[case["solver"]]
        return {"bytes": steps * (products * (matrix + dense) + vectors * 4 * rows),
                "flops": steps * (products * 2 * nnz + 2 * vectors * rows)}
    return {"bytes": matrix + dense, "flops": mul * nnz * width}


def tolerance(case):
    # about four times the distance from the 64-bit results: 1e-7 in float32
    # and complex64 (sums of any order), 2.1e-4 in float16, 1.7e-3 in bfloat16,
    # and 4e-6 for the iterate at which a solver stops
    if case["op"] == "solve":
        return {"rel": 2e-5}
    if case["dtype"] == "f16":
        return {"rel": 1e-3, "max": 5e-3}
    if case["dtype"] == "bf16":
        return {"rel": 8e-3, "max": 4e-2}
    return {"rel": 1e-6, "max": 4e-5}


# -- the same in 64 bits -----------------------------------------------------
def _wide(t):
    return t.to(torch.complex128 if t.is_complex() else torch.float64)


def _add_rows(out, at, terms):
    if out.is_complex():
        torch.view_as_real(out).index_add_(0, at, torch.view_as_real(terms))
    else:
        out.index_add_(0, at, terms)


class _Wide:
    """The matrix's products in 64 bits, over pieces of its values."""

    def __init__(self, data, indices, indptr, shape):
        self.data, self.cols, self.shape = _wide(data), indices.long(), shape
        self.rows = torch.repeat_interleave(
            torch.arange(shape[0], device=data.device), (indptr[1:] - indptr[:-1]).long())

    def _pieces(self, width):
        step = max(1, 100_000_000 // max(1, width))
        return range(0, self.data.numel(), step), step

    def times(self, x, transposed=False):
        take, put = (self.rows, self.cols) if transposed else (self.cols, self.rows)
        flat = x if x.ndim == 2 else x[:, None]
        out = torch.zeros(self.shape[1 if transposed else 0], flat.shape[1], dtype=flat.dtype,
                          device=flat.device)
        starts, step = self._pieces(flat.shape[1])
        for s in starts:
            e = s + step
            _add_rows(out, put[s:e], self.data[s:e, None] * flat[take[s:e]])
        return out if x.ndim == 2 else out[:, 0]

    def value_gradient(self, x, g):
        x, g = (t if t.ndim == 2 else t[:, None] for t in (x, g))
        out = torch.empty(self.data.numel(), dtype=x.dtype, device=x.device)
        starts, step = self._pieces(x.shape[1])
        for s in starts:
            e = s + step
            out[s:e] = (g[self.rows[s:e]] * x[self.cols[s:e]].conj()).sum(1)
        return out


def _cg(a, b, tol):
    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), r.dot(r)
    while rr.sqrt() > tol:
        ap = a.times(p)
        alpha = rr / p.dot(ap)
        x, r = x + alpha * p, r - alpha * ap
        new = r.dot(r)
        p, rr = r + new / rr * p, new
    return x


def _bicgstab(a, b, tol):
    x, r = torch.zeros_like(b), b.clone()
    hat, rho, p = r.clone(), r.dot(r), r.clone()
    while True:
        v = a.times(p)
        alpha = rho / hat.dot(v)
        s = r - alpha * v
        if s.norm() <= tol:
            return x + alpha * p
        t = a.times(s)
        omega = t.dot(s) / t.dot(t)
        x, r = x + alpha * p + omega * s, s - omega * t
        if r.norm() <= tol:
            return x
        new = hat.dot(r)
        p = r + new / rho * alpha / omega * (p - omega * v)
        rho = new


def _least_residual(a, b, tol, restart):
    """GMRES over cycles of ``restart`` steps, tested between them; with
    ``restart`` 0 one cycle tested at every step (the iterates of MINRES)."""
    x = torch.zeros_like(b)
    while True:
        r = b - a.times(x)
        beta = r.norm()
        if beta <= tol:
            return x
        basis, h = [r / beta], torch.zeros(201, 200, dtype=torch.float64)
        for j in range(restart or 200):
            w = a.times(basis[j])
            for _ in range(2):
                for i, q in enumerate(basis):
                    c = q.dot(w)
                    h[i, j] += c.item()
                    w = w - c * q
            h[j + 1, j] = w.norm().item()
            basis.append(w / w.norm())
            if restart and j + 1 < restart:
                continue
            e = torch.zeros(j + 2, 1, dtype=torch.float64)
            e[0] = beta.item()
            y = torch.linalg.lstsq(h[:j + 2, :j + 1], e).solution
            now = x + torch.stack(basis[:j + 1], 1) @ y[:, 0].to(b.device)
            if restart or (b - a.times(now)).norm() <= tol:
                break
        x = now


def exact(case, seed):
    data, indices, indptr, shape, operands = _inputs(case, seed)
    a = _Wide(data, indices, indptr, shape)
    op = case["op"]
    wide = [_wide(t) for t in operands]
    if op in ("spmv", "spmm"):
        return a.times(wide[0])
    if op == "batch":
        return a.times(wide[0].T.contiguous()).T.contiguous()
    if op == "adjoint":
        return a.times(wide[0], transposed=True)
    if op == "train":
        x, g = wide
        grads = (a.value_gradient(x, g),) if case["trained"] else ()
        return (a.times(x), *grads, a.times(g, transposed=True))
    b = wide[0]
    tol = 1e-5 * b.norm()
    if case["solver"] == "cg":
        x = _cg(a, b, tol)
    elif case["solver"] == "bicgstab":
        x = _bicgstab(a, b, tol)
    else:
        x = _least_residual(a, b, tol, 20 if case["solver"] == "gmres" else 0)
    return x, None
