"""The dataflow apply beyond its own tests: ops of many input segments (the
kernel's table takes 1024, read 64 at a time), applies of two trees at once, and
least-squares applies that are known to run it."""
import ctypes as C
import threading

import numpy as np
import pytest

import spaqr_public_amd as sq
from spaqr_public_amd import gen
from test_gpu_flow import BACK, PULL, SOLVE_T, WY, grid

pytestmark = pytest.mark.gpu
dp = C.POINTER(C.c_double)
EPS = np.finfo(float).eps


def run(ktest, pieces, kind, m, k, par, unit, A, B, n, x, xn):
    i, f = C.c_int, ktest.ktest_flow_pieces
    f.argtypes = [i, i, i, i, i, i, dp, i, dp, i, i, dp, dp, dp]
    A, B = (None if M is None else np.asfortranarray(M) for M in (A, B))
    out = np.full(m, np.nan)
    ptr = lambda M: None if M is None else M.ctypes.data_as(dp)
    ld = lambda M: 0 if M is None else M.shape[0]
    assert f(pieces, kind, m, k, par, unit, ptr(A), ld(A), ptr(B), ld(B), n, ptr(x), ptr(xn), ptr(out)) == 0
    return out


@pytest.mark.parametrize("m,k,rows,pieces", [(65, 20, 64, 65), (200, 40, 256, 129), (300, 33, 64, 64), (1024, 31, 64, 1024),
                                             (2000, 65, 128, 1000)])
def test_reflector_op_of_many_segments(ktest, m, k, rows, pieces):
    rng = np.random.default_rng(m + k)
    V = np.tril(rng.standard_normal((m, k)) / np.sqrt(m), -1) + np.eye(m, k)
    W = np.tril(rng.standard_normal((m, k)))
    x = rng.standard_normal(m)
    got = run(ktest, pieces, WY, m, k, rows, 1, V, W, 0, x, np.zeros(1))
    # two dot products, of m and of k terms
    bound = (m + k + 4) * EPS * (abs(x) + abs(W) @ (abs(V).T @ abs(x)))
    assert np.all(abs(got - (x - W @ (V.T @ x))) <= bound)


@pytest.mark.parametrize("k,n,parts,pieces", [(65, 40, 2, 65), (200, 90, 3, 130), (1024, 3, 1, 1024)])
def test_triangular_ops_of_many_segments(ktest, k, n, parts, pieces):
    rng = np.random.default_rng(k)
    R = np.triu(rng.standard_normal((k, k)) / k, 1) + np.diag(1.0 + rng.random(k))
    Bn, x, xn = rng.standard_normal((k, n)), rng.standard_normal(k), rng.standard_normal(n)
    tol = 20 * (k + n) * EPS  # R is well conditioned
    got = run(ktest, pieces, BACK, k, k, parts, 0, R, Bn, n, x, xn)
    size = np.linalg.norm(x) + np.linalg.norm(Bn) * np.linalg.norm(xn)
    assert np.linalg.norm(got - np.linalg.solve(R, x - Bn @ xn)) <= tol * size
    got = run(ktest, pieces, SOLVE_T, k, k, 1, 0, R, None, 0, x, np.zeros(1))
    assert np.linalg.norm(got - np.linalg.solve(R.T, x)) <= tol * np.linalg.norm(x)


@pytest.mark.parametrize("m,n,pieces", [(65, 70, 65), (300, 100, 200)])
def test_pull_op_of_many_segments(ktest, m, n, pieces):
    rng = np.random.default_rng(m)
    Bn, x, xn = rng.standard_normal((n, m)), rng.standard_normal(m), rng.standard_normal(n)
    got = run(ktest, pieces, PULL, m, 32, 1, 0, None, Bn, n, x, xn)
    bound = (n + 2) * EPS * (abs(x) + abs(Bn).T @ abs(xn))
    assert np.all(abs(got - (x - Bn.T @ xn)) <= bound)


def factored(A, n, d, tol, square=1):
    t = sq.Tree(sq.default_levels(A.shape[1]), 0, sq.FP64)
    t.set_scale(1)
    t.set_tol(tol)
    t.set_square(square)
    t.set_tensor_coordinates(n, d)
    t.kernel_timing(True)
    t.partition(A)
    t.assemble(A)
    t.factorize()
    t.flow = "wy" in t.kernel_stats()  # formed for the dataflow apply only
    t.kernel_timing(False)
    return t


def test_two_trees_at_once():
    trees = [factored(grid(n, d), n, d, tol) for n, d, tol in ((50, 2, 1e-6), (15, 3, 1e-1))]
    assert all(t.flow for t in trees)
    rng = np.random.default_rng(0)
    bs = [rng.standard_normal(t.n) for t in trees]
    want = [(t.solve(b), t.solve_transpose(b)) for t, b in zip(trees, bs)]
    differ = []
    start = threading.Barrier(2)

    def work(t, b, w):
        start.wait()
        for _ in range(40):
            if not (np.array_equal(t.solve(b), w[0]) and np.array_equal(t.solve_transpose(b), w[1])):
                differ.append(t)

    threads = [threading.Thread(target=work, args=a) for a in zip(trees, bs, want)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not differ  # sums in a fixed order, whatever else runs
    for t in trees:
        t.close()


@pytest.mark.parametrize("n", [16, 24, 40])
def test_least_squares_residual(monkeypatch, n):
    """At tol 0 the factors are those of A: x solves A^T A x = b."""
    A, _ = sq.colscale(gen.laplacian_gradient_ls(n, 1e-2))
    b = np.random.default_rng(n).standard_normal(A.shape[1])
    two = np.linalg.norm(A.toarray(), 2)**2
    # two solves with R, each of at most 50 steps in a row that are within a few
    # hundred eps of backward stable
    bar = 1e4 * EPS
    for reg, flow in (("0", False), ("1", True)):
        monkeypatch.setenv("SPAQR_REFL_REGISTER", reg)
        t = factored(A, n, 2, 0.0, square=0)
        assert t.flow == flow
        x = t.solve_nrml(b)
        assert np.linalg.norm(A.T @ (A @ x) - b) <= bar * two * np.linalg.norm(x)
        assert not flow or np.array_equal(t.solve_nrml(b), x)
        t.close()
