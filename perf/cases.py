"""The work that programs have this framework do, as measurable cases.

A case names a grid problem (edge ``n``, dimension ``d``), what is done with it (``kind``), and
the options of that call. The kinds, each through the package's public entry points:

* ``apply``: one preconditioner apply ``Tree.solve_device`` on ``nrhs`` device columns, the call
  that another program's Krylov loop makes once per iteration; the factorization is in hand.
  ``transpose`` applies the adjoint (``Tree.solve_transpose_device``). FP64 factors: an FP32
  factor is there to be corrected by the FP64 iteration, and is measured in the whole solves.
* ``direct``: the exact factorization of new values (every level skips the sparsification) and
  one solve, the use as a sparse direct solver.
* ``pcg``: ``Tree.factorize`` of new values and ``cg_device`` to 1e-12, the benchmark's step.
* ``gmres``: the same for a nonsymmetric matrix: PLU factorization, ``gmres_device`` to 1e-10.
* ``grad``: the differentiable solve: forward, adjoint, and the gradients of the cell
  coefficients and the right-hand sides.
* ``outer``: the gradient with respect to the stored values alone (``Matrix.sampled_outer_device``).

A program keeps the tree of its sparsity pattern (partition and symbolic assembly) and the
device copy of the matrix, so ``prepare`` makes them. Right-hand sides are N(0, 1);
``field = "kappa"`` problems have log-normal cell coefficients, drawn from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import spand_public_amd as S
from spand_public_amd.autograd import fv_solver, fv_values, sparse_solve
from spand_public_amd.problems import (DiffusionFV, auto_nlevels, convdiff, gaussian_field, linspace_nd, neglapl,
                                       seeded_rhs, symmetric_graph)

PECLET, VELOCITY = 10.0, (1.0, 0.5, 0.25)
CORRELATION = {2: 16.0, 3: 8.0}  # cells, of log kappa


def listed():
    return [
        # the smallest call: one column on a small 2D problem, where launches and latency count
        {"name": "apply_square40_f64", "kind": "apply", "n": 40, "d": 2, "nrhs": 1, "tol": 1e-2, "prec": "f64",
         "field": "laplace", "transpose": False},
        # one Krylov iteration's apply on the benchmark's problem, at its four columns
        {"name": "apply_cube64_f64", "kind": "apply", "n": 64, "d": 3, "nrhs": 4, "tol": 1e-2, "prec": "f64",
         "field": "laplace", "transpose": False},
        # a wide block of columns (the differentiable workload's 32) on its 512 x 512 grid
        {"name": "apply_square512_wide", "kind": "apply", "n": 512, "d": 2, "nrhs": 32, "tol": 1e-2,
         "prec": "f64", "field": "kappa", "transpose": False},
        # the adjoint apply of a nonsymmetric factorization, odd edge, odd column count
        {"name": "apply_convdiff37_t", "kind": "apply", "n": 37, "d": 3, "nrhs": 3, "tol": 1e-2, "prec": "f64",
         "field": "convdiff", "transpose": True},
        # a sparse direct solver in 2D, odd edge
        {"name": "direct_square201_f64", "kind": "direct", "n": 201, "d": 2, "nrhs": 1, "tol": 0.0, "prec": "f64",
         "field": "kappa"},
        # factor and solve of a small 3D problem, as one of many (the reference's test sizes)
        {"name": "pcg_cube15_f64", "kind": "pcg", "n": 15, "d": 3, "nrhs": 1, "tol": 1e-2, "prec": "f64",
         "field": "kappa"},
        # the benchmark's step, in both factor precisions
        {"name": "pcg_cube64_f32", "kind": "pcg", "n": 64, "d": 3, "nrhs": 4, "tol": 1e-2, "prec": "f32",
         "field": "laplace"},
        {"name": "pcg_cube64_f64", "kind": "pcg", "n": 64, "d": 3, "nrhs": 4, "tol": 1e-2, "prec": "f64",
         "field": "laplace"},
        # the largest: variable coefficients at the tighter tolerance
        {"name": "pcg_cube96_kappa_f32", "kind": "pcg", "n": 96, "d": 3, "nrhs": 4, "tol": 1e-3, "prec": "f32",
         "field": "kappa"},
        # nonsymmetric: PLU factorization and GMRES on eight columns
        {"name": "gmres_convdiff64_f32", "kind": "gmres", "n": 64, "d": 3, "nrhs": 8, "tol": 1e-2, "prec": "f32",
         "field": "convdiff"},
        # the differentiable workload: forward and backward on 32 columns
        {"name": "grad_square512_f64", "kind": "grad", "n": 512, "d": 2, "nrhs": 32, "tol": 1e-2, "prec": "f64",
         "field": "kappa"},
        # the values' gradient alone, as an inverse problem accumulates it over its snapshots
        {"name": "outer_square300", "kind": "outer", "n": 300, "d": 2, "nrhs": 16, "tol": 0.0, "prec": "f64",
         "field": "laplace"},
    ]


def _edge(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))


def draw(rng):
    kind = rng.choice(["apply", "apply", "direct", "pcg", "pcg", "gmres", "grad", "outer"])
    d = rng.choice([2, 3])
    case = {"kind": kind, "d": d, "tol": rng.choice([1e-1, 1e-2, 1e-3]), "prec": rng.choice(["f64", "f32"]),
            "field": rng.choice(["laplace", "kappa"]), "nrhs": rng.choice([1, 2, 3, 4, 7, 8, 16, 32])}
    case["n"] = _edge(rng, 24, 512) if d == 2 else _edge(rng, 9, 64)
    if kind == "apply":
        case.update(prec="f64", transpose=False)
        if rng.random() < 0.3:
            case["field"], case["transpose"] = "convdiff", rng.random() < 0.5
    elif kind == "direct":
        case.update(tol=0.0, prec="f64", n=_edge(rng, 24, 256) if d == 2 else _edge(rng, 9, 24))
    elif kind == "gmres":
        case.update(field="convdiff", nrhs=min(case["nrhs"], 8))
    elif kind == "grad":
        case.update(prec="f64", field="kappa", n=case["n"] if d == 2 else min(case["n"], 40))
    elif kind == "outer":
        case.update(tol=0.0, prec="f64", field="laplace")
    return case


# -- inputs -----------------------------------------------------------------------------


def _log_kappa(case, seed):
    # sigma 2 and 1: the workloads' contrasts in 3D and 2D
    return gaussian_field(case["n"], case["d"], 2.0 if case["d"] == 3 else 1.0, CORRELATION[case["d"]], seed)


def _matrix(case, seed):
    n, d = case["n"], case["d"]
    if case["field"] == "kappa":
        return DiffusionFV(n, d).matrix(np.exp(_log_kappa(case, seed)))
    return convdiff(n, d, PECLET, VELOCITY) if case["field"] == "convdiff" else neglapl(n, d)


def _rows(case, seed):
    """The right-hand sides, one row per column of the block: (nrhs, N) in device memory."""
    return torch.from_numpy(np.ascontiguousarray(seeded_rhs(case["n"] ** case["d"], case["nrhs"], seed).T)).cuda()


def _tree(case, A):
    t = S.Tree(max(2, auto_nlevels(A.n)))
    t.set_use_geo(True)
    t.set_Xcoo(linspace_nd(case["n"], case["d"]))
    t.set_tol(case["tol"])
    t.set_precision(S.FP32 if case["prec"] == "f32" else S.FP64)
    if case["field"] == "convdiff":
        t.set_symm_kind("GEN")
    if case["kind"] == "direct":
        t.set_skip(t.get_nlevels())
    t.partition(symmetric_graph(A))
    t.assemble(A)
    return t


def prepare(case, seed):
    n, d, kind = case["n"], case["d"], case["kind"]
    state = {"case": case, "b": _rows(case, seed)}
    if kind == "grad":
        fv = DiffusionFV(n, d)
        state["fv"] = fv
        state["solver"] = fv_solver(fv, max(2, auto_nlevels(fv.N)), tol=case["tol"])
        state["kappa"] = torch.from_numpy(np.exp(_log_kappa(case, seed))).cuda()
        state["target"] = torch.from_numpy(seeded_rhs(fv.N, case["nrhs"], seed + 1)).cuda()
        state["b"] = state["b"].t().contiguous()
        return state
    A = _matrix(case, seed)
    if kind == "outer":
        state["matrix"] = S.Matrix(A)
        state["v"] = _rows(case, seed + 1)
        state["out"] = torch.zeros(A.nnz, dtype=torch.float64, device="cuda")
        return state
    state["tree"] = _tree(case, A)
    state["x"] = torch.zeros_like(state["b"])
    if kind == "apply":
        state["tree"].factorize()
    else:
        state["matrix"] = S.Matrix(A)
        state["vals"] = torch.from_numpy(A.nzval).cuda()
    return state


# -- one pass ---------------------------------------------------------------------------


def run(state):
    case, b = state["case"], state["b"]
    kind = case["kind"]
    if kind == "grad":
        kappa = state["kappa"].detach().requires_grad_(True)
        bb = b.detach().requires_grad_(True)
        x = sparse_solve(fv_values(state["fv"], kappa), bb, state["solver"])
        (0.5 * (x - state["target"]).square().sum()).backward()
        return {"x": x.detach(), "dkappa": kappa.grad, "db": bb.grad}
    nrhs, N = b.shape
    if kind == "outer":
        state["matrix"].sampled_outer_device(b.data_ptr(), state["v"].data_ptr(), nrhs, N, -1.0,
                                             state["out"].data_ptr())
        return state["out"]
    tree, x, stream = state["tree"], state["x"], torch.cuda.current_stream().cuda_stream
    if kind != "apply":
        vals = state["vals"]
        tree.assemble_values_device(vals.data_ptr(), vals.numel(), stream)
        tree.factorize()
    if kind in ("apply", "direct"):
        x.copy_(b)
        solve = tree.solve_transpose_device if case.get("transpose") else tree.solve_device
        solve(x.data_ptr(), nrhs, N, stream)
        return x
    x.zero_()
    state["matrix"].set_values_device(vals.data_ptr(), vals.numel(), stream)
    if kind == "pcg":
        _, info = S.cg_device(state["matrix"], tree, b.data_ptr(), x.data_ptr(), nrhs, N, iters=500, tol=1e-12)
    else:
        _, info = S.gmres_device(state["matrix"], tree, b.data_ptr(), x.data_ptr(), nrhs, N, iters=500, restart=30,
                                 tol=1e-10)
    if info["status"] != 0:
        raise RuntimeError("the Krylov solve did not converge")
    return x


# -- what a pass cannot do without ------------------------------------------------------


def _stored(case):
    """About the stored factor's entries: measured per unknown, for the tolerances in use."""
    N = case["n"] ** case["d"]
    return N * (80 if case["d"] == 2 else 295)


def work(case):
    n, d, r = case["n"], case["d"], case["nrhs"]
    N = n ** d
    nnz = N + 2 * d * (n - 1) * n ** (d - 1)
    vectors = 8 * N * r
    if case["kind"] == "apply":  # the factor, the columns in and out
        e = _stored(case)
        return {"bytes": e * (4 if case["prec"] == "f32" else 8) + 2 * vectors, "flops": 4 * e * r}
    if case["kind"] == "outer":
        return {"bytes": 12 * nnz + 2 * vectors, "flops": 2 * nnz * r}
    # the values and their pattern, the columns in and out; the factor is a result of the path itself
    bytes_, flops = 12 * nnz + 2 * vectors, 2 * nnz * r
    return {"bytes": 2 * bytes_, "flops": 2 * flops} if case["kind"] == "grad" else {"bytes": bytes_, "flops": flops}


# -- the same results in plain torch, 64 bits -------------------------------------------



def _diffusion(kappa, d):
    """u -> A u on (nrhs, n, .., n) blocks for cell coefficients (n, .., n), and A's diagonal."""
    n = kappa.shape[0]
    faces = []
    diag = torch.zeros_like(kappa)
    for ax in range(d):
        ka, kb = kappa.narrow(ax, 0, n - 1), kappa.narrow(ax, 1, n - 1)
        t = 2.0 * ka * kb / (ka + kb)
        faces.append(t)
        diag.narrow(ax, 0, n - 1).add_(t)
        diag.narrow(ax, 1, n - 1).add_(t)
        diag.narrow(ax, 0, 1).add_(kappa.narrow(ax, 0, 1))
        diag.narrow(ax, n - 1, 1).add_(kappa.narrow(ax, n - 1, 1))

    def apply(u):
        y = diag * u
        for ax, t in enumerate(faces):
            y.narrow(ax + 1, 0, n - 1).sub_(t * u.narrow(ax + 1, 1, n - 1))
            y.narrow(ax + 1, 1, n - 1).sub_(t * u.narrow(ax + 1, 0, n - 1))
        return y

    return apply, diag


def _convection(n, d, transpose):
    """The same for ``convdiff``: the neighbour behind along each axis carries the flow."""
    diag = torch.full((n,) * d, 2.0 * d + PECLET * sum(VELOCITY[:d]), dtype=torch.float64, device="cuda")

    def apply(u):
        y = diag * u
        for ax in range(d):
            behind, ahead = 1.0 + PECLET * VELOCITY[ax], 1.0
            if transpose:
                behind, ahead = ahead, behind
            y.narrow(ax + 1, 1, n - 1).sub_(behind * u.narrow(ax + 1, 0, n - 1))
            y.narrow(ax + 1, 0, n - 1).sub_(ahead * u.narrow(ax + 1, 1, n - 1))
        return y

    return apply, diag


def _dot(a, b):
    return (a * b).flatten(1).sum(1).reshape((-1,) + (1,) * (a.dim() - 1))


def _cg(apply, diag, b):
    """Jacobi-preconditioned conjugate gradients until the residual stops falling."""
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz = z.clone(), _dot(r, z)
    size = _dot(b, b).sqrt()
    for i in range(40000):
        q = apply(p)
        a = rz / _dot(p, q)
        x += a * p
        r -= a * q
        z = r / diag
        new = _dot(r, z)
        p = z + (new / rz) * p
        rz = new
        if i % 50 == 49 and bool(((_dot(r, r).sqrt() / size) < 1e-15).all()):
            break
    return x


def _bicgstab(apply, diag, b):
    x, r = torch.zeros_like(b), b.clone()
    r0, p = r.clone(), r.clone()
    rho, size = _dot(r0, r), _dot(b, b).sqrt()
    for i in range(5000):
        ph = p / diag
        v = apply(ph)
        a = rho / _dot(r0, v)
        s = r - a * v
        sh = s / diag
        t = apply(sh)
        w = _dot(t, s) / _dot(t, t)
        x += a * ph + w * sh
        r = s - w * t
        if bool(((_dot(r, r).sqrt() / size) < 1e-11).all()):
            break
        new = _dot(r0, r)
        p = r + (new / rho) * (a / w) * (p - w * v)
        rho = new
    return x


def _refined(solve, apply, diag, b):
    x = solve(apply, diag, b)
    for _ in range(2):
        r = b - apply(x)
        x = x + solve(apply, diag, r)
    return x


def exact(case, seed):
    n, d, kind = case["n"], case["d"], case["kind"]
    if kind == "apply":
        return None  # an approximate inverse: the tolerance's own, with no value besides it
    grid = (n,) * d
    b = _rows(case, seed)
    r = case["nrhs"]
    if kind == "outer":
        v = _rows(case, seed + 1).reshape((r,) + grid)
        u = b.reshape((r,) + grid)
        # entry (i, j), by column j and then row i: the neighbours of j in the order of their index
        stack = torch.full(grid + (2 * d + 1,), float("nan"), dtype=torch.float64, device="cuda")
        stack[..., d] = -(u * v).sum(0)
        for ax in range(d):
            stack.narrow(ax, 1, n - 1)[..., ax] = -(u.narrow(ax + 1, 0, n - 1) * v.narrow(ax + 1, 1, n - 1)).sum(0)
            stack.narrow(ax, 0, n - 1)[..., 2 * d - ax] = -(u.narrow(ax + 1, 1, n - 1)
                                                            * v.narrow(ax + 1, 0, n - 1)).sum(0)
        flat = stack.reshape(-1)
        return flat[~torch.isnan(flat)]
    b = b.reshape((r,) + grid)
    if case["field"] == "convdiff":
        apply, diag = _convection(n, d, False)
        return _refined(_bicgstab, apply, diag, b).reshape(r, -1)
    kappa = torch.ones(grid, dtype=torch.float64, device="cuda")
    if case["field"] == "kappa":
        kappa = torch.from_numpy(np.exp(_log_kappa(case, seed)).reshape(grid)).cuda()
    apply, diag = _diffusion(kappa, d)
    x = _refined(_cg, apply, diag, b)
    if kind != "grad":
        return x.reshape(r, -1)
    target = torch.from_numpy(seeded_rhs(n ** d, r, seed + 1)).cuda().t().reshape((r,) + grid)
    lam = _refined(_cg, apply, diag, x - target)
    # dL/dkappa = -lam . (dA/dkappa) x, with A a sum over faces
    k = kappa.clone().requires_grad_(True)
    energy = torch.zeros((), dtype=torch.float64, device="cuda")
    for ax in range(d):
        ka, kb = k.narrow(ax, 0, n - 1), k.narrow(ax, 1, n - 1)
        dx, dl = torch.diff(x, dim=ax + 1), torch.diff(lam, dim=ax + 1)
        energy = energy - (2.0 * ka * kb / (ka + kb) * (dx * dl).sum(0)).sum()
        for at in (0, n - 1):
            energy = energy - (k.narrow(ax, at, 1) * (x * lam).sum(0).narrow(ax, at, 1)).sum()
    energy.backward()
    return {"x": x.reshape(r, -1).t(), "dkappa": k.grad.reshape(-1), "db": lam.reshape(r, -1).t()}
