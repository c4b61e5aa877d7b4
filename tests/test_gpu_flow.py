"""The dataflow apply: single ops at the edges of its tiles (32 columns, 64-row
chunks, parts that exchange their sums, several tiles per wave) against dense
products and solves, and whole trees against the staged program."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import spaqr_public_amd as sq

pytestmark = pytest.mark.gpu
dp, fp = C.POINTER(C.c_double), C.POINTER(C.c_float)
WY, BACK, SOLVE_T, PULL = range(4)


def run(ktest, f32, kind, m, k, par, unit, A, B, n, x, xn):
    """A, B: Fortran-ordered or None."""
    tp, f = (fp, ktest.ktest_flow_f32) if f32 else (dp, ktest.ktest_flow)
    i = C.c_int
    f.argtypes = [i, i, i, i, i, tp, i, tp, i, i, dp, dp, dp]
    t = np.float32 if f32 else np.float64
    A, B = (None if M is None else np.asfortranarray(M, dtype=t) for M in (A, B))
    out = np.full(m, np.nan)
    ptr = lambda M: None if M is None else M.ctypes.data_as(tp)
    ld = lambda M: 0 if M is None else max(M.shape[0], 1)
    x, xn = np.ascontiguousarray(x, float), np.ascontiguousarray(xn, float)
    assert f(kind, m, k, par, unit, ptr(A), ld(A), ptr(B), ld(B), n, x.ctypes.data_as(dp), xn.ctypes.data_as(dp),
             out.ctypes.data_as(dp)) == 0
    return out


def eps_of(f32):
    return np.finfo(np.float32 if f32 else np.float64).eps


def rounded(M, f32):
    return M.astype(np.float32).astype(float) if f32 else M


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("m,k,rows", [(1, 1, 64), (31, 31, 64), (33, 32, 64), (64, 64, 64), (65, 33, 64), (100, 65, 64),
                                      (128, 97, 128), (129, 128, 64), (193, 129, 128), (256, 20, 256), (257, 32, 256),
                                      (300, 160, 64), (700, 40, 1024), (1000, 1000, 64), (1024, 1024, 1024),
                                      (2000, 31, 64)])
def test_reflector_op(ktest, f32, m, k, rows):
    rng = np.random.default_rng(m + k)
    # what lies outside the trapezoids is never used: V shares its panel with
    # R, W's upper part is not written
    V, W = rng.standard_normal((m, k)) / np.sqrt(m), rng.standard_normal((m, k))
    up = np.triu_indices(m, 0, k)
    V[up], W[np.triu_indices(m, 1, k)] = np.nan, np.nan
    x = rounded(rng.standard_normal(m), f32)
    Vd = rounded(np.where(np.tri(m, k, -1) > 0, V, 0.0), f32) + np.eye(m, k)
    Wd = rounded(np.where(np.tri(m, k) > 0, W, 0.0), f32)
    for unit, (A, B), (Ad, Bd) in ((1, (V, W), (Vd, Wd)), (0, (W, V), (Wd, Vd))):
        got = run(ktest, f32, WY, m, k, rows, unit, A, B, 0, x, np.zeros(1))
        # two dot products, of m and of k terms: |error| <= (m + k) eps |B| |A|^T |x|
        bound = (m + k + 4) * eps_of(f32) * (abs(x) + abs(Bd) @ (abs(Ad).T @ abs(x)))
        assert np.all(abs(got - (x - Bd @ (Ad.T @ x))) <= bound)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("k,n,parts", [(1, 0, 1), (20, 7, 1), (32, 40, 2), (33, 300, 3), (64, 65, 1), (65, 200, 4),
                                       (129, 100, 2), (193, 700, 8), (290, 64, 2), (600, 90, 2), (1024, 3, 1)])
def test_triangular_ops(ktest, f32, k, n, parts):
    rng = np.random.default_rng(k + n)
    R = rng.standard_normal((k, k)) / k
    R[np.diag_indices(k)] = 1.0 + rng.random(k)
    R[np.tril_indices(k, -1)] = np.nan  # V lies there
    Bn = rng.standard_normal((k, max(n, 1)))
    x, xn = rounded(rng.standard_normal(k), f32), rounded(rng.standard_normal(max(n, 1)), f32)
    Rd, Bd = rounded(np.triu(np.nan_to_num(R)), f32), rounded(Bn, f32)[:, :n]
    # R is well conditioned (diagonal 1..2, rows of others of norm < 1): a
    # backward stable solve errs by a small multiple of k eps in norm
    tol = 20 * (k + n) * eps_of(f32)
    want = np.linalg.solve(Rd, x - Bd @ xn[:n])
    got = run(ktest, f32, BACK, k, k, parts, 0, R, Bn if n else None, n, x, xn)
    size = np.linalg.norm(x) + np.linalg.norm(Bd) * np.linalg.norm(xn[:n])
    assert np.linalg.norm(got - want) <= tol * size
    want = np.linalg.solve(Rd.T, x)
    got = run(ktest, f32, SOLVE_T, k, k, 1, 0, R, None, 0, x, np.zeros(1))
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(x)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("m,n", [(1, 1), (31, 7), (32, 71), (33, 8), (65, 300), (200, 72), (300, 1000)])
def test_pull_op(ktest, f32, m, n):
    rng = np.random.default_rng(m + n)
    Bn = rng.standard_normal((n, m))
    x, xn = rounded(rng.standard_normal(m), f32), rounded(rng.standard_normal(n), f32)
    Bd = rounded(Bn, f32)
    got = run(ktest, f32, PULL, m, 32, 1, 0, None, Bn, n, x, xn)
    bound = (n + 2) * eps_of(f32) * (abs(x) + abs(Bd).T @ abs(xn))
    assert np.all(abs(got - (x - Bd.T @ xn)) <= bound)


def grid(n, d):
    L = sp.diags([-1, 2.2, -0.9], [-1, 0, 1], shape=(n, n))
    A = L
    for _ in range(d - 1):
        A = sp.kron(A, sp.identity(n)) + sp.kron(sp.identity(A.shape[0]), L)
    return A.tocsc()


@pytest.mark.parametrize("n,d,precision,tol", [(5, 2, 8, 1e-2), (16, 2, 8, 0.0), (30, 2, 4, 1e-3), (50, 2, 8, 1e-6),
                                               (9, 3, 8, 0.0), (14, 3, 4, 1e-2), (17, 3, 8, 1e-1)])
def test_against_staged_program(monkeypatch, n, d, precision, tol):
    A = grid(n, d)
    b = np.random.default_rng(n).standard_normal(A.shape[0])
    got = []
    for reg in ("0", "1"):
        monkeypatch.setenv("SPAQR_REFL_REGISTER", reg)
        t = sq.Tree(sq.default_levels(A.shape[1]) if n > 8 else 2, 0, precision)
        t.set_scale(1)
        t.set_tol(tol)
        t.set_square(1)
        t.set_tensor_coordinates(n, d)
        t.partition(A)
        t.assemble(A)
        t.factorize()
        got.append([t.solve(b), t.solve_transpose(b), t.solve(b)])
        t.close()
    # the same product of at most 50 orthogonal and well-conditioned triangular
    # factors (grid operators, condition below 1e3), each within a few hundred
    # eps of the exact one
    eps = np.finfo(np.float32 if precision == 4 else np.float64).eps
    for a, c in zip(*got):
        assert np.linalg.norm(a - c) <= 1e4 * eps * np.linalg.norm(a)
    assert np.array_equal(got[1][0], got[1][2])  # no order of arrival in the sums


@pytest.mark.parametrize("n,precision,tol", [(16, 8, 1e-2), (24, 8, 0.0), (40, 4, 1e-2), (57, 8, 1e-1)])
def test_least_squares_against_staged_program(monkeypatch, n, precision, tol):
    from spaqr_public_amd import gen
    A, _ = sq.colscale(gen.laplacian_gradient_ls(n, 1e-2))
    b = np.random.default_rng(n).standard_normal(A.shape[1])
    got = []
    for reg in ("0", "1"):
        monkeypatch.setenv("SPAQR_REFL_REGISTER", reg)
        t = sq.Tree(sq.default_levels(A.shape[1]), 0, precision)
        t.set_scale(1)
        t.set_tol(tol)
        t.set_square(0)
        t.set_tensor_coordinates(n, 2)
        t.partition(A)
        t.assemble(A)
        t.factorize()
        got.append([t.solve_nrml(b), t.solve_nrml(b)])
        t.close()
    # R^{-1} R^{-T} b by two routes, each backward stable; the column-scaled
    # matrix with its regularising rows has a condition below 1e4, squared here
    eps = np.finfo(np.float32 if precision == 4 else np.float64).eps
    for a, c in zip(*got):
        assert np.linalg.norm(a - c) <= (1e8 if precision == 8 else 1e5) * eps * np.linalg.norm(a)
    assert precision == 4 or np.array_equal(got[1][0], got[1][1])
