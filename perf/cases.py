"""Workloads of the library as a user's program runs them, through its public entry points.

Five kinds, each over grid sides from a few dozen to the benchmark's 64^3 (2-D: up to 256^2):

  flow    a new matrix: partition, assemble, factorize, upload, Krylov solve to 1e-12 on device vectors
          (the benchmark's path, from the matrix on).  Least-squares trees end in CGLS instead of GMRES.
  gmres   another right-hand side on a tree that is kept: GMRES to 1e-12 on device vectors
  apply   one preconditioner apply x = M^-1 b on a kept tree, for a caller that runs its own Krylov method
          (adjoint: x = M^-T b)
  grad    the differentiable solve on a kept solver: x = A^-1 b, then the gradients for b and for A's values

The right-hand sides are A x_true for a random x_true, so that the solutions are known.  The advection-diffusion
matrices have a rough reaction coefficient and a velocity drawn from the seed; the sizes, the stencils and the
tolerances are those of the benchmark's workloads (2-D: 1e-3, 3-D: 1e-2).
"""
import math

import numpy as np
import torch

import spaqr_public_amd as sq
from spaqr_public_amd import autograd as sg
from spaqr_public_amd import gen

RES = 1e-12      # GMRES and refinement tolerance, the benchmark's
RES_LS = 1e-13   # CGLS: its stopping quantity is that of the normal equations


def listed():
    return [
        # the smallest systems: a caller that factors a small 2-D problem and solves once; latency and launches count
        dict(name="flow2d_40", kind="flow", matrix="advdiff", dim=2, n=40, precision="fp64"),
        # the size of the published 2-D run (128^2)
        dict(name="flow2d_128", kind="flow", matrix="advdiff", dim=2, n=128, precision="fp64"),
        # a small 3-D problem with an odd side
        dict(name="flow3d_15", kind="flow", matrix="advdiff", dim=3, n=15, precision="fp64"),
        # an ordinary 3-D problem with an odd side
        dict(name="flow3d_33", kind="flow", matrix="advdiff", dim=3, n=33, precision="fp64"),
        # the benchmark's size (64^3): factorization, large interfaces
        dict(name="flow3d_64", kind="flow", matrix="advdiff", dim=3, n=64, precision="fp64"),
        # the mixed form: FP32 factors, FP64 refinement
        dict(name="flow3d_45_mixed", kind="flow", matrix="advdiff", dim=3, n=45, precision="fp32"),
        # high-contrast diffusion: more iterations, other ranks
        dict(name="contrast3d_32", kind="flow", matrix="contrast", dim=3, n=32, precision="fp64"),
        # least squares (Laplacian and gradient rows), CGLS
        dict(name="ls2d_100", kind="flow", matrix="ls", dim=2, n=100, precision="fp64"),
        # time stepping or several loads: many right-hand sides on one factorization
        dict(name="gmres3d_40", kind="gmres", matrix="advdiff", dim=3, n=40, precision="fp64"),
        # the preconditioner inside a caller's own Krylov method: small, and large
        dict(name="apply2d_64", kind="apply", matrix="advdiff", dim=2, n=64, precision="fp64", adjoint=False),
        dict(name="apply3d_52", kind="apply", matrix="advdiff", dim=3, n=52, precision="fp64", adjoint=False),
        # forward and backward of the differentiable solve, an instance of the adjoint batch (2-D, side 64..256)
        dict(name="grad2d_150", kind="grad", matrix="advdiff", dim=2, n=150, precision="fp64"),
    ]


def _side(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "flow", "flow", "gmres", "apply", "grad"])
    if kind == "grad":
        return dict(kind=kind, matrix="advdiff", dim=2, n=_side(rng, 64, 256), precision="fp64")
    if kind == "apply":
        dim = rng.choice([2, 3, 3])
        return dict(kind=kind, matrix="advdiff", dim=dim, n=_side(rng, 32, 256) if dim == 2 else _side(rng, 12, 60),
                    precision="fp64", adjoint=rng.random() < 0.5)
    matrix = rng.choice(["advdiff", "advdiff", "contrast", "ls"]) if kind == "flow" else "advdiff"
    precision = rng.choice(["fp64", "fp64", "fp32"])
    if matrix == "ls":
        return dict(kind=kind, matrix=matrix, dim=2, n=_side(rng, 32, 128), precision="fp64")
    if matrix == "contrast":
        return dict(kind=kind, matrix=matrix, dim=3, n=_side(rng, 16, 48), precision=precision)
    dim = rng.choice([2, 3, 3])
    return dict(kind=kind, matrix=matrix, dim=dim, n=_side(rng, 32, 256) if dim == 2 else _side(rng, 12, 60),
                precision=precision)


# ---- what a pass cannot do without ----------------------------------------

# unknowns: GFLOP of the factorization (LAWN 41 counts of its dense steps), MB of its factors, MB one apply reads
_SIZES = {
    2: ((1024, 0.06, 1.6, 2.4), (4096, 0.29, 7.4, 10.8), (16384, 1.31, 31.5, 46.2), (65536, 5.75, 131.1, 193.5)),
    3: ((1728, 0.33, 4.1, 7.0), (4096, 1.66, 12.2, 21.8), (13824, 13.36, 56.5, 103.6), (35937, 62.18, 179.2, 321.5),
        (110592, 351.94, 637.9, 1244.6), (262144, 1244.0, 1708.6, 3426.6)),
    "ls": ((2304, 0.27, 7.1, 10.0), (16384, 5.28, 71.7, 107.9)),
}


def _sizes(key, unknowns):
    rows = _SIZES[key]
    lx = [math.log(r[0]) for r in rows]
    k = min(max(sum(v < math.log(unknowns) for v in lx) - 1, 0), len(rows) - 2)
    w = (math.log(unknowns) - lx[k]) / (lx[k + 1] - lx[k])
    return [math.exp((1 - w) * math.log(rows[k][j]) + w * math.log(rows[k + 1][j])) for j in (1, 2, 3)]


def work(case):
    unknowns = case["n"] ** case["dim"]
    nnz = (2 * case["dim"] + 1) * unknowns * (2 if case["matrix"] == "ls" else 1)
    gflop, factor_mb, apply_mb = _sizes("ls" if case["matrix"] == "ls" else case["dim"], unknowns)
    wide = 1.0 if case["precision"] == "fp64" else 0.5
    factor, apply_, matrix = factor_mb * 1e6 * wide, apply_mb * 1e6 * wide, 12.0 * nnz
    its = {"ls": 20, "contrast": 13}.get(case["matrix"], 6 if case["dim"] == 2 else 10)
    krylov = its * (apply_ + matrix)
    krylov_flops = its * (apply_ / (4 * wide) + 2 * nnz)
    if case["kind"] == "flow":
        return dict(bytes=matrix + factor + krylov, flops=gflop * 1e9 + krylov_flops)
    if case["kind"] == "gmres":
        return dict(bytes=krylov, flops=krylov_flops)
    if case["kind"] == "grad":
        return dict(bytes=2 * krylov, flops=2 * krylov_flops)
    return dict(bytes=apply_ + 16.0 * unknowns, flops=apply_ / 4)


# ---- inputs ----------------------------------------------------------------

def _solution(case, seed):
    return np.random.default_rng([seed, 1]).standard_normal(case["n"] ** case["dim"])


def _adjoint_solution(case, seed):
    return np.random.default_rng([seed, 2]).standard_normal(case["n"] ** case["dim"])


def _matrix(case, seed):
    """The caller's matrix (CSC, sorted row indices)."""
    rng = np.random.default_rng([seed, 0])
    n, dim = case["n"], case["dim"]
    if case["matrix"] == "contrast":
        return gen.high_contrast_diffusion(n, dim, 8, int(rng.integers(1 << 30)))
    if case["matrix"] == "ls":
        A = gen.laplacian_gradient_ls(n, 1e-2)
        A.data *= 1.0 + 0.05 * rng.random(A.nnz)
        return A
    speed = 1000.0 if dim == 2 else 100.0
    A = gen.advection_diffusion(n, dim, 1.0, list(speed * rng.uniform(0.3, 1.0, dim)))
    A.setdiag(A.diagonal() + rng.uniform(0.0, 100.0, A.shape[0]))
    return A


def _device(v):
    return torch.as_tensor(np.ascontiguousarray(v), dtype=torch.float64, device="cuda")


def _new_tree(case, A):
    t = sq.Tree(sq.default_levels(A.shape[1]), 0, sq.FP64 if case["precision"] == "fp64" else sq.FP32)
    t.set_scale(1)
    t.set_tol(1e-3 if case["dim"] == 2 and case["matrix"] != "ls" else 1e-2)
    t.set_order(1.0)
    t.set_square(0 if case["matrix"] == "ls" else 1)
    t.set_tensor_coordinates(case["n"], case["dim"])
    t.set_phase_sync(0)
    t.partition(A)
    t.assemble(A)
    t.factorize()
    return t


def prepare(case, seed):
    A = _matrix(case, seed)
    x_true = _solution(case, seed)
    if case["kind"] == "grad":
        w = _device(A.T @ _adjoint_solution(case, seed))
        solver = sg.SparseSolver(A.indptr, A.indices, A.data, case["n"], case["dim"], tol=1e-3, res=RES)
        return dict(case=case, solver=solver, w=w, values=_device(A.data).requires_grad_(),
                    b=_device(A @ x_true).requires_grad_())
    As, _ = sq.colscale(A)  # the driver's column scaling
    b = _device(As @ x_true)
    state = dict(case=case, A=As, b=b, x=torch.zeros(As.shape[1], dtype=torch.float64, device="cuda"))
    if case["kind"] != "flow":
        state["tree"] = _new_tree(case, As)
        state["M"] = sq.Matrix(state["tree"], As)
    torch.cuda.synchronize()
    return state


# ---- one pass ----------------------------------------------------------------

def _krylov(case, tree, M, b, x):
    x.zero_()
    torch.cuda.current_stream().synchronize()  # the tree works on a stream of its own
    if case["matrix"] == "ls":
        sq.cgls_device(tree, M, b.data_ptr(), x.data_ptr(), tol=RES_LS)
    else:
        sq.gmres_device(tree, M, b.data_ptr(), x.data_ptr(), tol=RES)


def run(state):
    case = state["case"]
    if case["kind"] == "grad":
        x = sg.solve(state["values"], state["b"], state["solver"])
        dvalues, db = torch.autograd.grad((x * state["w"]).sum(), (state["values"], state["b"]))
        return dict(x=x.detach(), dvalues=dvalues, db=db)
    b, x = state["b"], state["x"]
    if case["kind"] == "flow":
        tree = _new_tree(case, state["A"])
        M = sq.Matrix(tree, state["A"])
        _krylov(case, tree, M, b, x)
        M.close()
        tree.close()
    elif case["kind"] == "gmres":
        _krylov(case, state["tree"], state["M"], b, x)
    elif case["adjoint"]:
        state["tree"].solve_transpose_device(b.data_ptr(), x.data_ptr())
    else:
        state["tree"].solve_device(b.data_ptr(), x.data_ptr())
    return x


# ---- the same in 64 bits -----------------------------------------------------

def exact(case, seed):
    if case["kind"] == "apply":
        return None  # M approximates A to the tolerance: it has no value of its own
    x = _solution(case, seed)
    if case["kind"] != "grad":
        return x
    # L = w . x with w = A^T lam: dL/db = lam, dL/dA_ij = -lam_i x_j on the 5-point pattern, column by column
    lam, n = _adjoint_solution(case, seed), case["n"]
    j = np.arange(n * n)
    at = np.stack([j - n, j - 1, j, j + 1, j + n], axis=1)
    there = np.stack([j >= n, j % n > 0, j >= 0, j % n < n - 1, j < n * (n - 1)], axis=1)
    col = np.broadcast_to(j[:, None], at.shape)
    return dict(x=x, dvalues=-lam[at[there]] * x[col[there]], db=lam)
