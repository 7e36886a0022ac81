"""Timed cases of the CSR5 path: what a program built on it spends its time in.

The products (one and several right-hand sides, FP64 and FP32, stencil,
irregular and power-law matrices, A and A^T), the conjugate-gradient solvers
(one, several right-hand sides, a batch of uneven systems with its gradients)
and the conversion of a CSR matrix that is already on the GPU. Matrices are
made on the GPU from the seed; structured grids keep their pattern and draw
new coefficients, the others draw both.
"""
from __future__ import annotations

import math

import torch

from diploma_research_amd import Csr5, conjugate_gradient, conjugate_gradient_multi
from diploma_research_amd.autograd import solve

DEV = "cuda"


# ------------------------------------------------------------------- cases --

def listed():
    return [
        # the smallest call: a 5-point operator of 64 x 64 cells (the size of
        # a smoke run, or of the coarse level of a solver), where launches and
        # the host path count
        dict(name="spmv-2d-64", kind="spmv", grid="64x64", coef=0.0, sigma=5, f32=False),
        # the product of a structured-grid solver: 7-point Poisson, 128^3
        dict(name="spmv-3d-128", kind="spmv", grid="128x128x128", coef=0.0, sigma=7, f32=False),
        # the same kind of operator with variable coefficients on a ragged
        # grid, multiplied in FP32 (a preconditioner or an inner solver)
        dict(name="spmv-3d-ragged-f32", kind="spmv", grid="131x97x119", coef=1.0, sigma=7, f32=True),
        # a general matrix (mesh-like band, uneven rows, some empty, a few
        # long) at the default tile height, assembled on the GPU
        dict(name="spmv-irregular", kind="irregular", rows=700001, cols=700001, mean=12, band=4000, empty=0.02,
             sigma=16, f32=False),
        # a graph: Pareto row lengths, columns all over a large x, in the
        # column-sliced form that large scattered matrices are kept in
        dict(name="spmv-powerlaw", kind="powerlaw", n=2100000, sigma=8, f32=False),
        # several right-hand sides as a program holds them in torch
        # (row-major n x k): 8 load cases on a 3-D grid
        dict(name="spmm-3d-k8", kind="spmm", grid="112x112x112", coef=1.0, sigma=7, k=8, cols_major=False,
             f32=False),
        # the transposed product of a rectangular matrix (least squares,
        # adjoints of non-symmetric operators)
        dict(name="transpose-irregular", kind="transpose", rows=300007, cols=200003, mean=14, band=9000, empty=0.01,
             sigma=16, f32=False),
        # a matrix assembled on the GPU by a program that changes its pattern
        # (adaptive meshes, contact): conversion and the first product
        dict(name="convert-irregular", kind="convert", rows=400009, cols=400009, mean=16, band=6000, empty=0.0,
             sigma=16, f32=False),
        # conjugate gradients on the 2-D 5-point operator of 256 x 256 cells:
        # iterations of a few microseconds
        dict(name="cg-2d-256", kind="cg", grid="256x256", coef=0.0, sigma=5, k=1, refined=False, rtol=1e-12),
        # conjugate gradients on the 128^3 Poisson operator, FP64
        dict(name="cg-3d-128", kind="cg", grid="128x128x128", coef=0.0, sigma=7, k=1, refined=False, rtol=1e-12),
        # 8 right-hand sides, FP32 iteration inside FP64 residual replacement,
        # variable coefficients
        dict(name="cg-multi-refined-64", kind="cg", grid="64x64x64", coef=1.0, sigma=7, k=8, refined=True,
             rtol=1e-12),
        # a batch of uneven 2-D diffusion systems solved under autograd, with
        # the gradients of the matrix values and of the right-hand sides
        dict(name="solve-batch-grad", kind="solve", systems=16, side_min=60, side_max=300, coef=1.0, sigma=5,
             rtol=1e-12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid3(rng, lo, hi):
    """A ragged 3-D grid of about lo^3 to hi^3 cells, no side over hi."""
    s = _log_int(rng, lo, hi)
    return "x".join(str(max(3, int(s * rng.uniform(0.75, 1.0)))) for _ in range(3))


def _grid2(rng, lo, hi):
    s = _log_int(rng, lo, hi)
    return "x".join(str(max(3, int(s * rng.uniform(0.75, 1.0)))) for _ in range(2))


def draw(rng):
    kind = rng.choice(["spmv", "spmv", "irregular", "powerlaw", "spmm", "spmm", "transpose", "convert", "cg", "cg",
                       "cg", "solve"])
    coef = rng.choice([0.0, 1.0])
    if kind == "spmv":
        if rng.random() < 0.5:
            return dict(kind=kind, grid=_grid2(rng, 24, 1500), coef=coef, sigma=rng.choice([5, 5, 10, 16]),
                        f32=rng.random() < 0.4)
        return dict(kind=kind, grid=_grid3(rng, 10, 140), coef=coef, sigma=rng.choice([7, 7, 8, 16]),
                    f32=rng.random() < 0.4)
    if kind in ("irregular", "transpose", "convert"):
        rows = _log_int(rng, 2000, 700001 if kind == "irregular" else 300007)
        cols = rows if kind != "transpose" else _log_int(rng, max(1000, rows // 3), rows)
        return dict(kind=kind, rows=rows, cols=cols, mean=rng.randint(4, 16), band=_log_int(rng, 200, 10000),
                    empty=rng.choice([0.0, 0.01, 0.05]), sigma=rng.choice([8, 16, 16]),
                    f32=kind != "convert" and rng.random() < 0.3)
    if kind == "powerlaw":
        return dict(kind=kind, n=_log_int(rng, 300000, 2100000), sigma=rng.choice([4, 8]), f32=rng.random() < 0.3)
    if kind == "spmm":
        return dict(kind=kind, grid=_grid3(rng, 16, 100), coef=coef, sigma=rng.choice([7, 7, 16]),
                    k=rng.choice([2, 3, 4, 5, 6, 8, 8, 11, 16]), cols_major=rng.random() < 0.5,
                    f32=rng.random() < 0.4)
    if kind == "cg":
        k = rng.choice([1, 1, 2, 3, 5, 8])
        two = rng.random() < 0.5
        return dict(kind=kind, grid=_grid2(rng, 24, 256 if k == 1 else 128) if two else _grid3(rng, 8, 128 if k == 1 else 48),
                    coef=coef, sigma=5 if two else 7, k=k, refined=k > 1 and rng.random() < 0.4, rtol=1e-12)
    lo = rng.randint(20, 60)
    return dict(kind="solve", systems=rng.randint(2, 16), side_min=lo, side_max=_log_int(rng, lo + 20, 240), coef=coef,
                sigma=5, rtol=1e-12)


# ------------------------------------------------------------------ inputs --

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _uniform(g, n):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * 2 - 1


def _shape(case):
    return tuple(int(s) for s in case["grid"].split("x"))


def _stencil(shape, coef, g):
    """Dirichlet diffusion operator on a structured grid: (row_ptr, cols,
    vals). coef is the log-normal spread of the cells' diffusivity (0: the
    Poisson operator); faces take the harmonic mean of their two cells."""
    n, dims = math.prod(shape), len(shape)
    if coef:
        kap = torch.exp(coef * torch.randn(shape, generator=g, device=DEV, dtype=torch.float64))
    else:
        kap = torch.ones(shape, device=DEV, dtype=torch.float64)
    # one slot per neighbour, in column order: -axis 0, ..., diagonal, ..., +axis 0
    slots = 2 * dims + 1
    val = torch.zeros((slots, *shape), device=DEV, dtype=torch.float64)
    off = torch.zeros(slots, device=DEV, dtype=torch.int64)
    has = torch.zeros((slots, *shape), device=DEV, dtype=torch.bool)
    has[dims] = True
    stride = n
    for ax in range(dims):
        stride //= shape[ax]
        m = shape[ax]
        k1, k2 = kap.narrow(ax, 0, m - 1), kap.narrow(ax, 1, m - 1)
        face = 2 * k1 * k2 / (k1 + k2)
        for slot, start in ((ax, 1), (slots - 1 - ax, 0)):
            val[slot].narrow(ax, start, m - 1).copy_(-face)
            has[slot].narrow(ax, start, m - 1).fill_(True)
        off[ax], off[slots - 1 - ax] = -stride, stride
        val[dims].narrow(ax, 0, m - 1).add_(face)
        val[dims].narrow(ax, 1, m - 1).add_(face)
        val[dims].narrow(ax, 0, 1).add_(kap.narrow(ax, 0, 1))
        val[dims].narrow(ax, m - 1, 1).add_(kap.narrow(ax, m - 1, 1))
    has = has.reshape(slots, n).t()
    cols = (torch.arange(n, device=DEV)[:, None] + off[None, :])[has]
    vals = val.reshape(slots, n).t()[has]
    return _row_ptr(has.sum(1)), cols.to(torch.int32), vals


def _row_ptr(lens):
    rp = torch.zeros(lens.numel() + 1, device=DEV, dtype=torch.int64)
    torch.cumsum(lens, 0, out=rp[1:])
    return rp.to(torch.int32)


def _from_keys(key, rows, cols, g):
    """CSR of sorted, distinct keys row*cols + col, with normal values."""
    key = torch.unique(key)
    r = torch.div(key, cols, rounding_mode="floor")
    rp = _row_ptr(torch.bincount(r, minlength=rows))
    vals = torch.randn(key.numel(), generator=g, device=DEV, dtype=torch.float64)
    return rp, (key - r * cols).to(torch.int32), vals


def _irregular(case, g):
    """Mesh-like rows: lengths spread around the mean, some rows empty, a few
    over 50 times the mean, columns within a band around the scaled diagonal."""
    rows, cols, mean = case["rows"], case["cols"], case["mean"]
    lens = torch.randint(1, 2 * mean, (rows,), generator=g, device=DEV)
    lens[torch.rand(rows, generator=g, device=DEV) < case["empty"]] = 0
    lens[torch.randint(0, rows, (max(1, rows // 100000),), generator=g, device=DEV)] = 60 * mean
    r = torch.repeat_interleave(torch.arange(rows, device=DEV), lens)
    at = r * cols // rows + ((torch.rand(r.numel(), generator=g, device=DEV, dtype=torch.float64) - 0.5) *
                             2 * case["band"]).to(torch.int64)
    return _from_keys(r * cols + at.clamp_(0, cols - 1), rows, cols, g)


def _powerlaw(case, g):
    """Pareto row lengths (shape 2, scale 8, at most 10000: about 15.5 per
    row), columns uniform."""
    n = case["n"]
    u = 1.0 - torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    lens = torch.floor(8.0 / torch.sqrt(u)).to(torch.int64).clamp_(1, 10000)
    r = torch.repeat_interleave(torch.arange(n, device=DEV), lens)
    return _from_keys(r * n + torch.randint(0, n, (r.numel(),), generator=g, device=DEV), n, n, g)


def _sides(case):
    """The grids of a batch: evenly spread widths, heights 3/4 of them."""
    s, lo, hi = case["systems"], case["side_min"], case["side_max"]
    return [(max(3, w * 3 // 4), w) for w in (lo + (hi - lo) * i // max(1, s - 1) for i in range(s))]


def _host(csr):
    return tuple(t.cpu().numpy() for t in csr)


def _product(csr, x, rows):
    """A x in 64 bits (x: one column or several), with torch alone."""
    rp, ci, v = csr
    r = torch.repeat_interleave(torch.arange(rows, device=DEV), (rp[1:] - rp[:-1]).to(torch.int64))
    if x.dim() == 1:
        return torch.zeros(rows, device=DEV, dtype=torch.float64).index_add_(0, r, v * x[ci.long()])
    return torch.stack([torch.zeros(rows, device=DEV, dtype=torch.float64).index_add_(0, r, v * x[ci.long(), j])
                        for j in range(x.shape[1])], 1)


def _inputs(case, seed):
    """The matrix (CSR on the GPU) and the vectors of a case."""
    g, kind = _gen(seed), case["kind"]
    if kind == "solve":
        mats = [_stencil(s, case["coef"], g) for s in _sides(case)]
        x = [_uniform(g, m[0].numel() - 1) for m in mats]
        lam = [_uniform(g, m[0].numel() - 1) for m in mats]
        return dict(mats=mats, x=x, lam=lam)
    if kind in ("spmv", "spmm", "cg"):
        shape = _shape(case)
        csr, rows = _stencil(shape, case["coef"], g), math.prod(shape)
        cols = rows
    elif kind == "powerlaw":
        csr, rows, cols = _powerlaw(case, g), case["n"], case["n"]
    else:
        csr, rows, cols = _irregular(case, g), case["rows"], case["cols"]
    k = case.get("k", 1)
    n = rows if kind == "transpose" else cols
    x = _uniform(g, n * k).reshape((n, k) if k > 1 else (n,))
    return dict(csr=csr, rows=rows, cols=cols, x=x.to(torch.float32) if case.get("f32") else x)


def _vector(case, x):
    """x as the program holds it: several columns row-major, or one after another."""
    return x.t().contiguous().t() if case.get("cols_major") else x


# ------------------------------------------------------- the program's part --

def prepare(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    if kind == "solve":
        A = Csr5.from_csr_batched([(m[0].numel() - 1, *_host(m)) for m in d["mats"]], sigma=case["sigma"])
        b = torch.cat([_product(m, x, x.numel()) for m, x in zip(d["mats"], d["x"])])
        w = torch.cat([_product(m, x, x.numel()) for m, x in zip(d["mats"], d["lam"])])
        vals = torch.cat([m[2] for m in d["mats"]])
        return dict(case=case, A=A, vals=vals.requires_grad_(), b=b.requires_grad_(), w=w)
    csr, rows, cols = d["csr"], d["rows"], d["cols"]
    x = _vector(case, d["x"])
    if kind == "convert":
        return dict(case=case, csr=csr, x=x)
    if kind in ("irregular", "transpose"):
        A = Csr5.from_csr_device(rows, cols, *csr, sigma=case["sigma"], keep_f32=case["f32"])
    else:
        A = Csr5.from_csr((rows, cols, *_host(csr)), sigma=case["sigma"],
                          keep_f32=bool(case.get("f32") or case.get("refined")), xcd_slices=kind == "powerlaw")
    if kind == "cg":
        return dict(case=case, A=A, b=_product(csr, x, rows).contiguous())
    y = torch.empty(cols if kind == "transpose" else rows, dtype=x.dtype, device=DEV) if kind != "spmm" else None
    return dict(case=case, A=A, x=x, y=y)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("spmv", "irregular", "powerlaw"):
        return state["A"].spmv(state["x"], state["y"])
    if kind == "spmm":
        return state["A"].spmm(state["x"])
    if kind == "transpose":
        return state["A"].spmv_transpose(state["x"], state["y"])
    if kind == "convert":
        A = Csr5.from_csr_device(case["rows"], case["cols"], *state["csr"], sigma=case["sigma"])
        return A.spmv(state["x"])
    if kind == "cg":
        if case["k"] == 1:
            return conjugate_gradient(state["A"], state["b"], rtol=case["rtol"], max_iters=20000)[0]
        return conjugate_gradient_multi(state["A"], state["b"], rtol=case["rtol"], max_iters=20000,
                                        precision="f32-refined" if case["refined"] else "f64")[0]
    x = solve(state["A"], state["vals"], state["b"], rtol=case["rtol"], max_iters=20000)
    gv, gb = torch.autograd.grad(x, [state["vals"], state["b"]], state["w"])
    return dict(x=x, grad_vals=gv, grad_b=gb)


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    if kind == "solve":
        # b = A x and dL/dx = A lam, so the solution is x, dL/db = lam and
        # dL/da_ij = -lam_i x_j
        gv = [-lam[torch.repeat_interleave(torch.arange(x.numel(), device=DEV), (m[0][1:] - m[0][:-1]).long())] *
              x[m[1].long()] for m, x, lam in zip(d["mats"], d["x"], d["lam"])]
        return dict(x=torch.cat(d["x"]), grad_vals=torch.cat(gv), grad_b=torch.cat(d["lam"]))
    if kind == "cg":
        return d["x"]  # b = A x
    csr, rows, x = d["csr"], d["rows"], d["x"].double()
    if kind == "transpose":
        rp, ci, v = csr
        r = torch.repeat_interleave(torch.arange(rows, device=DEV), (rp[1:] - rp[:-1]).long())
        return torch.zeros(d["cols"], device=DEV, dtype=torch.float64).index_add_(0, ci.long(), v * x[r])
    return _product(csr, x, rows)


def _stencil_nnz(shape):
    n = math.prod(shape)
    return n + sum(2 * (n // s) * (s - 1) for s in shape)


def _iterations(shape, coef, rtol):
    """About the conjugate-gradient iterations to rtol: the Poisson
    operator's condition grows with the square of the longest side;
    log-normal coefficients take about three times as many steps."""
    return int(0.42 * 0.5 * (0.64 * (max(shape) + 1)) * math.log(2 / rtol) * (3 if coef else 1)) + 1


def work(case):
    """Bytes and operations of one pass: (value + 4-byte column) per stored
    element, the vectors once per product; a solver's iteration reads the
    matrix and the direction and passes over its vectors ten times in all."""
    kind = case["kind"]
    vb = 4 if case.get("f32") else 8
    if kind == "solve":
        nbytes = flops = 0
        for s in _sides(case):
            n, nnz, it = math.prod(s), _stencil_nnz(s), 2 * _iterations(s, case["coef"], case["rtol"])
            nbytes += it * (12 * nnz + 80 * n)
            flops += it * (2 * nnz + 10 * n)
        return dict(bytes=nbytes, flops=flops)
    if kind == "cg":
        s, k, vb = _shape(case), case["k"], 4 if case["refined"] else 8
        n, nnz, it = math.prod(s), _stencil_nnz(s), _iterations(s, case["coef"], case["rtol"])
        return dict(bytes=it * ((vb + 4) * nnz + 10 * k * vb * n), flops=it * k * (2 * nnz + 10 * n))
    if kind in ("spmv", "spmm"):
        s = _shape(case)
        rows = cols = math.prod(s)
        nnz = _stencil_nnz(s)
    elif kind == "powerlaw":
        rows = cols = case["n"]
        nnz = int(15.5 * rows)
    else:
        rows, cols = case["rows"], case["cols"]
        nnz = int(rows * case["mean"] * (1 - case["empty"]))
    k = case.get("k", 1)
    nbytes = (vb + 4) * nnz + vb * k * (rows + cols)
    if kind == "convert":  # the CSR arrays in, the converted ones out, then the product
        nbytes += 2 * (12 * nnz + 4 * rows)
    return dict(bytes=nbytes, flops=2 * k * nnz)
