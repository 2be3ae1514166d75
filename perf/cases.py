"""Workloads the SpMV framework is timed on, through its public entry points.

A case is a plain dict:

  op         what one pass does, as a user's program calls it
               run       y = A x                       (engine.launch)
               run_x     y' = A' x' in Kr numbering    (engine.launch_x)
               residual  r = b - A x                   (engine.residual)
               newton    new matrix values, then the residual: one step of a
                         nonlinear solver (engine.update_values + residual)
               train     new matrix values, the product, and its two gradients
                         (engine.update_values + launch + backward)
               scan      a new sparsity pattern already on the device becomes an
                         engine and is multiplied once (engine.from_device + launch)
               batch     many mixed matrices in one launch (batch.run)
  mesh, n    finite-element problem and grid size (warpkernel_amd.fe)
  dtype      matrix values: f64, or f32 (FP32 x, FP64 y)
  variant    1 (WPK1) or 2 (WPK2 with `threshold`)
  k          right-hand sides; the block vectors are row-major [n, k]
  strided    the block vectors are columns of a wider array
"""
import math
import random

import numpy as np
import torch

from warpkernel_amd import batch, engine, fe, structure, structure2

MESHES = ("laplace2d", "diffusion", "elastic", "tets", "tets_perm")


def _case(name, op, mesh, n, **kw):
    c = dict(name=name, op=op, mesh=mesh, n=n, dtype="f64", variant=1, threshold=0, k=1, strided=False)
    c.update(kw)
    return c


def listed():
    return [
        # a 2D Poisson solver's product: 16.6K rows, everything in cache, bound by latency
        _case("laplace2d_128_run", "run", "laplace2d", 128),
        # a 3D elasticity solver's product at full size (the benchmark's headline matrix)
        _case("elastic_64_run", "run", "elastic", 64),
        # the same solver on a coarser level, split rows, vectors kept in Kr numbering
        _case("elastic_32_wpk2_run_x", "run_x", "elastic", 32, variant=2, threshold=27),
        # an unstructured tetrahedral mesh, numbered in grid order
        _case("tets_96_run", "run", "tets", 96),
        # the same mesh numbered at random, as a mesh generator may leave it
        _case("tets_96_perm_run", "run", "tets_perm", 96),
        # block Krylov / eigenvalue iterations: 16 vectors on a coarse level
        _case("elastic_32_k16", "run", "elastic", 32, k=16),
        # many load cases at once on a larger elasticity matrix
        _case("elastic_48_k32", "run", "elastic", 48, k=32),
        # mixed-precision smoother: FP32 matrix and vectors, compensated sums, 8 vectors
        _case("elastic_32_f32_k8", "run", "elastic", 32, dtype="f32", k=8),
        # a differentiable PDE layer's training step: new coefficients, forward, both gradients
        _case("diffusion_48_train", "train", "diffusion", 48),
        # a nonlinear elasticity step: reassembled values, then the residual
        _case("elastic_48_newton", "newton", "elastic", 48),
        # remeshing: a device CSR becomes a layout and is used
        _case("elastic_40_scan", "scan", "elastic", 40),
        # a multi-domain program: many small and medium matrices in one launch
        _case("batch_24_k1", "batch", "mix", 24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["run", "run", "run", "run_x", "residual", "train", "newton", "scan", "batch"])
    if op == "batch":
        return dict(op=op, mesh="mix", n=rng.randint(4, 24), dtype=rng.choice(["f64", "f64", "f32"]), variant=1,
                    threshold=0, k=rng.choice([1, 1, 2, 4, 8]), strided=False)
    mesh = rng.choice(MESHES)
    k = 1 if op in ("scan", "newton") or rng.random() < 0.4 else rng.choice([2, 3, 4, 5, 7, 8, 11, 12, 16, 24, 32])
    # the grid's largest side keeps every draw at or below the largest listed case
    top = {"laplace2d": 1000, "diffusion": 100, "elastic": 64, "tets": 96, "tets_perm": 96}[mesh]
    if k > 1 or op in ("train", "newton", "scan"):
        top = {"laplace2d": 600, "diffusion": 60, "elastic": 40, "tets": 60, "tets_perm": 40}[mesh]
    n = _log_int(rng, {"laplace2d": 24, "elastic": 5}.get(mesh, 8), top)
    dtype = "f32" if op in ("run", "run_x", "scan") and rng.random() < 0.25 else "f64"
    variant = 2 if op != "train" and rng.random() < 0.25 else 1
    threshold = {"laplace2d": 4, "diffusion": 9, "elastic": 27, "tets": 5, "tets_perm": 5}[mesh] if variant == 2 else 0
    strided = k > 1 and op != "train" and rng.random() < 0.2
    return dict(op=op, mesh=mesh, n=n, dtype=dtype, variant=variant, threshold=threshold, k=k, strided=strided)


# ------------------------------------------------------------------- inputs
def _mix(count):
    """Grids of `count` mixed matrices: 2D Laplacians (True) and 3D elasticity,
    sizes log-uniform from 2K to 100K rows."""
    rng = random.Random(1004)
    grids = []
    for _ in range(count):
        rows = math.exp(rng.uniform(math.log(2000), math.log(100000)))
        two = rng.random() < 0.5
        grids.append((two, round(math.sqrt(rows)) - 1 if two else round((rows / 3) ** (1 / 3)) - 1))
    return grids


def _matrices(case, seed):
    # the meshes are the case's, the coefficients (and a random numbering) the seed's
    n = case["n"]
    if case["mesh"] == "mix":
        make2, make3 = fe.q1_laplace_2d, fe.hex_elastic_3d
        return [(make2 if two else make3)(g, seed=31 * seed + i) for i, (two, g) in enumerate(_mix(n))]
    make = {
        "laplace2d": lambda: fe.q1_laplace_2d(n, seed=11 + 7 * seed),
        "diffusion": lambda: fe.hex_laplace_3d(n, seed=12 + 7 * seed),
        "elastic": lambda: fe.hex_elastic_3d(n, seed=13 + 7 * seed),
        "tets": lambda: fe.tet_poisson_3d(n, seed=14 + 7 * seed),
        "tets_perm": lambda: fe.tet_poisson_3d(n, seed=14 + 7 * seed, perm_seed=16 + 7 * seed),
    }[case["mesh"]]
    return [make()]


def _vector(rows, k, seed, dtype=np.float64):
    v = np.random.default_rng(seed).uniform(-1.0, 1.0, (rows, k)).astype(dtype)
    return v[:, 0] if k == 1 else v


def _inputs(case, seed):
    """Host inputs of one pass: the matrices, x per matrix, and what else the op reads."""
    ms = _matrices(case, seed)
    xdt = np.float32 if case["dtype"] == "f32" else np.float64
    k = case["k"]
    inp = dict(ms=ms, xs=[_vector(m.ncols, k, 1000 * seed + 17 + i, xdt) for i, m in enumerate(ms)])
    m = ms[0]
    if case["op"] in ("residual", "newton"):
        inp["b"] = _vector(m.nrows, k, 1000 * seed + 501)
    if case["op"] in ("newton", "train"):
        # the coefficients of the next step: each row's entries scaled by its own factor
        scale = np.random.default_rng(1000 * seed + 502).lognormal(0.0, 0.2, m.nrows)
        inp["vals"] = m.vals * np.repeat(scale, m.row_lengths())
    if case["op"] == "train":
        inp["gy"] = _vector(m.nrows, k, 1000 * seed + 503)
    return inp


def _dev(v, strided=False):
    t = torch.from_numpy(np.ascontiguousarray(v)).cuda()
    if strided and t.dim() == 2:
        wide = torch.zeros((t.shape[0], t.shape[1] + 5), dtype=t.dtype, device="cuda")
        wide[:, : t.shape[1]] = t
        return wide[:, : t.shape[1]]
    return t


def _out(rows, case):
    return _dev(np.zeros((rows, case["k"]) if case["k"] > 1 else rows), case["strided"])


def _structure(case, m):
    if case["variant"] == 2:
        return structure2(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind, case["threshold"])
    return structure(64).scan(m.nnz, m.nrows, m.vals, m.rowptr, m.colind)


def prepare(case, seed):
    inp = _inputs(case, seed)
    m, op = inp["ms"][0], case["op"]
    if op == "scan":
        return dict(case=case, rowptr=_dev(m.rowptr), colind=_dev(m.colind), vals=_dev(m.vals),
                    x=_dev(inp["xs"][0], case["strided"]), y=_out(m.nrows, case))
    engs = [engine(_structure(case, a), a.vals, a.colind, dtype=case["dtype"], kr=op == "run_x",
                   adjoint=op == "train") for a in inp["ms"]]
    if op == "batch":
        xs = [_dev(x) for x in inp["xs"]]
        ys = [_out(a.nrows, case) for a in inp["ms"]]
        b = batch(engs)
        b.bind(xs, ys)
        return dict(case=case, batch=b, ys=ys)
    eng = engs[0]
    x = inp["xs"][0]
    if op == "run_x":
        x = x[eng.kernel.row_map]  # x' in Kr numbering
    st = dict(case=case, eng=eng, x=_dev(x, case["strided"]), y=_out(m.nrows, case))
    for key in ("b", "vals", "gy"):
        if key in inp:
            st[key] = _dev(inp[key], case["strided"])
    if op == "train":
        st["dx"], st["dvals"] = _out(m.ncols, case), _dev(np.zeros(m.nnz))
    return st


# --------------------------------------------------------------------- pass
def run(state):
    op = state["case"]["op"]
    if op == "batch":
        state["batch"].run()
        return state["ys"]
    if op == "scan":
        c = state["case"]
        eng = engine.from_device(state["rowptr"], state["colind"], state["vals"], variant=c["variant"],
                                 threshold=c["threshold"], dtype=c["dtype"])
        eng.launch(state["x"], state["y"])
        return state["y"]
    eng, x, y = state["eng"], state["x"], state["y"]
    if op == "run":
        eng.launch(x, y)
    elif op == "run_x":
        eng.launch_x(x, y)
    elif op == "residual":
        eng.residual(state["b"], x, y)
    elif op == "newton":
        eng.update_values(state["vals"])
        eng.residual(state["b"], x, y)
    else:
        eng.update_values(state["vals"])
        eng.launch(x, y)
        eng.backward(state["gy"], x, state["dx"], state["dvals"])
        return y, state["dx"], state["dvals"]
    return y


def _sizes(case):
    """(rows, nnz) of each matrix, as the grid gives them."""
    n = case["n"]
    grid = {
        "laplace2d": lambda g: ((g + 1) ** 2, (3 * g + 1) ** 2),
        "diffusion": lambda g: ((g + 1) ** 3, (3 * g + 1) ** 3),
        "elastic": lambda g: (3 * (g + 1) ** 3, 9 * (3 * g + 1) ** 3),
    }
    if case["mesh"] == "mix":
        return [grid["laplace2d" if two else "elastic"](g) for two, g in _mix(n)]
    if case["mesh"] in grid:
        return [grid[case["mesh"]](n)]
    # Kuhn tetrahedra: every node, and two entries per edge (few edges lose all their elements)
    edges = 3 * n * (n + 1) ** 2 + 3 * n * n * (n + 1) + n ** 3
    return [((n + 1) ** 3, (n + 1) ** 3 + 2 * edges)]


def work(case):
    op, k = case["op"], case["k"]
    s = 8 if case["dtype"] == "f64" else 4
    total, flops = 0, 0
    for rows, nnz in _sizes(case):
        total += nnz * (s + 4) + k * rows * (s + 8)
        flops += 2 * nnz * k
        if op in ("residual", "newton"):
            total += k * rows * 8
        if op == "newton":
            total += nnz * s  # the layout's values, written
        if op == "train":
            # values written to both layouts; the transposed pattern, gy, dx and the value gradient
            total += 2 * nnz * s + nnz * 4 + k * rows * 16 + nnz * 8
            flops += 4 * nnz * k
        if op == "scan":
            total += nnz * (8 - s) + rows * 4 + nnz * (s + 4)  # the CSR read, the padded arrays written
    return {"bytes": total, "flops": flops}


# -------------------------------------------------------------------- exact
def _product(m, vals, x):
    a = torch.sparse_csr_tensor(torch.from_numpy(m.rowptr), torch.from_numpy(m.colind), torch.from_numpy(vals),
                                size=(m.nrows, m.ncols), dtype=torch.float64)
    xt = torch.from_numpy(np.ascontiguousarray(x, dtype=np.float64).reshape(m.ncols, -1))
    y = (a @ xt).numpy()
    return y[:, 0] if x.ndim == 1 else y


def exact(case, seed):
    inp = _inputs(case, seed)
    op = case["op"]
    out = []
    for m, x in zip(inp["ms"], inp["xs"]):
        vals = inp.get("vals", m.vals)
        if case["dtype"] == "f32":
            vals = vals.astype(np.float32).astype(np.float64)
        y = _product(m, vals, x)
        if op in ("residual", "newton"):
            y = inp["b"] - y
        elif op == "run_x":
            y = y[np.argsort(-m.row_lengths(), kind="stable")]
        elif op == "train":
            rows = np.repeat(np.arange(m.nrows), m.row_lengths())
            gy, k = inp["gy"].reshape(m.nrows, -1), case["k"]
            x2 = x.reshape(m.ncols, -1)
            dx = np.stack([np.bincount(m.colind, weights=vals * gy[rows, j], minlength=m.ncols) for j in range(k)], 1)
            dv = sum(gy[rows, j] * x2[m.colind, j] for j in range(k))
            return y, (dx[:, 0] if x.ndim == 1 else dx), dv
        out.append(y)
    return out if op == "batch" else out[0]
