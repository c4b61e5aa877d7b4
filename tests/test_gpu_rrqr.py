"""Blocked truncated pivoted QR (rounds of a 64-candidate panel and a matrix-core
update) against the oracle's geqp3: ranks, pivot order and R, at the edges of
the panel forms (rows 16, 32, 48, 64, 112, 160, 224, 288, 384, 512, 704; up to
48 one wave for launches of many problems, else four), of
the update's row tiles and of its 32-column tiles, with exact ties, duplicate
and zero columns, and for both storage types."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def run(K, Cmat, tol, dtype=np.float64, nd=1):
    k, N = Cmat.shape
    ct = C.c_double if dtype == np.float64 else C.c_float
    f = K.ktest_rrqr if dtype == np.float64 else K.ktest_rrqr_f32
    tp, ip = C.POINTER(ct), C.POINTER(C.c_int)
    f.argtypes = [C.c_int, C.c_int, tp, tp, tp, C.c_double, C.c_int, ip, ip]
    Ct = np.asfortranarray(Cmat.T.astype(dtype))
    V = np.zeros((k, k), dtype=dtype, order="F")
    tau = np.zeros(k, dtype=dtype)
    perm = np.zeros(N, dtype=np.int32)
    rounds = C.c_int(0)
    rank = f(k, N, Ct.ctypes.data_as(tp), V.ctypes.data_as(tp), tau.ctypes.data_as(tp), tol, nd,
             perm.ctypes.data_as(ip), C.byref(rounds))
    assert rank >= 0
    return rank, Ct[:, :rank].T.astype(float), V[:, :rank].astype(float), tau[:rank].astype(float), perm[:rank], rounds.value


def q_apply(V, tau, M):
    """H_r ... H_1 M."""
    M = M.copy()
    for i in range(len(tau)):
        v = V[:, i].copy()
        v[:i] = 0.0
        v[i] = 1.0
        M -= np.outer(tau[i] * v, v @ M)
    return M


def graded(k, N, decay, seed):
    rng = np.random.default_rng(seed)
    r = min(k, N)
    U = np.linalg.qr(rng.standard_normal((k, k)))[0][:, :r]
    return (U * np.logspace(0, -decay, r)) @ rng.standard_normal((r, N))


FORMS = [(1, 1, 1e-2), (1, 70, 1e-2), (16, 63, 1e-10), (17, 64, 1e-10), (32, 65, 1e-3), (33, 31, 1e-10),
         (48, 700, 1e-3), (49, 257, 1e-3), (64, 1000, 1e-2), (65, 200, 1e-10), (112, 1500, 1e-2), (113, 40, 1e-10),
         (128, 333, 1e-2), (129, 161, 1e-2), (160, 900, 1e-2), (161, 2000, 1e-2), (192, 97, 1e-10), (193, 512, 1e-3),
         (224, 800, 1e-2), (225, 100, 1e-10), (288, 3000, 1e-2), (289, 600, 1e-2), (321, 500, 1e-3),
         (385, 700, 1e-2), (512, 900, 1e-2), (513, 650, 1e-2), (704, 1000, 1e-2)]


@pytest.mark.parametrize("k,N,tol,nd", [f + (1,) for f in FORMS] + [f + (1000,) for f in FORMS if f[0] <= 48])
def test_rrqr_forms(ktest, oracle, k, N, tol, nd):
    Cmat = graded(k, N, 4, 1000 * k + N)
    oracle.set_backend("own")
    Rref, jpvt, tau_ref = oracle.geqp3(np.asfortranarray(Cmat))
    rank_ref = oracle.choose_rank(np.diag(Rref)[:min(k, N)], tol)
    rank, R, V, tau, perm, rounds = run(ktest, Cmat, tol, nd=nd)
    assert rank == rank_ref
    assert np.array_equal(perm, jpvt[:rank])
    # backward error of r <= 704 Householder steps: a small multiple of r eps |C|
    scale = np.linalg.norm(Cmat)
    bar = 20 * max(rank, 1) * EPS * scale
    full = q_apply(V, tau, Cmat)
    want = full[:rank].copy()
    for p, j in enumerate(perm):
        want[p + 1:, j] = 0.0
    assert np.linalg.norm(R - want) <= bar
    assert np.linalg.norm(np.abs(R[np.arange(rank), perm]) - np.abs(np.diag(Rref)[:rank])) <= bar
    # what was cut off is below the rank test's bar: the next pivot norm
    if rank < min(k, N):
        assert np.max(np.linalg.norm(full[rank:], axis=0)) <= tol * abs(Rref[0, 0]) * (1 + 1e-12) + bar
    # a round finds at least one pivot, and one more round may only see the stop
    assert rounds <= rank + 1


# integer data with exact ties: norms and products are exact, so the order of
# the pivots is decided by positions alone
@pytest.mark.parametrize("nd", [1, 1000])
@pytest.mark.parametrize("k,N,seed", [(8, 300, 0), (20, 500, 1), (40, 3000, 2), (70, 1000, 3)])
def test_rrqr_ties(ktest, oracle, k, N, seed, nd):
    rng = np.random.default_rng(seed)
    Cmat = np.zeros((k, N))
    Cmat[rng.integers(0, k, N), np.arange(N)] = rng.choice([-2.0, 2.0, 1.0], N)  # scaled unit vectors
    Cmat[:, rng.choice(N, N // 10, replace=False)] = 0.0
    oracle.set_backend("own")
    Rref, jpvt, _ = oracle.geqp3(np.asfortranarray(Cmat))
    rank_ref = oracle.choose_rank(np.diag(Rref)[:min(k, N)], 1e-3)
    rank, R, V, tau, perm, _ = run(ktest, Cmat, 1e-3, nd=nd)
    assert rank == rank_ref
    assert np.array_equal(perm, jpvt[:rank])


@pytest.mark.parametrize("k,N", [(30, 0), (5, 200), (64, 64)])
def test_rrqr_degenerate(ktest, k, N):
    rank, R, V, tau, perm, _ = run(ktest, np.zeros((k, max(N, 1)))[:, :N], 1e-2)
    # a zero matrix: |r_00| = 0 and the test of step 1 is 0 / 0
    assert rank == (0 if N == 0 else 1)
    assert not np.any(tau)


# FP32 storage: R and the reflectors carry the storage rounding of every round
@pytest.mark.parametrize("k,N", [(20, 300), (100, 1200), (300, 700)])
def test_rrqr_f32(ktest, k, N):
    Cmat = graded(k, N, 3, k).astype(np.float32).astype(float)
    rank, R, V, tau, perm, rounds = run(ktest, Cmat, 1e-2, np.float32)
    assert rank > 0
    want = q_apply(V, tau, Cmat)[:rank]
    for p, j in enumerate(perm):
        want[p + 1:, j] = 0.0
    # each of at most `rank` reflectors is orthogonal to float rounding
    assert np.linalg.norm(R - want) <= rank * np.finfo(np.float32).eps * np.linalg.norm(Cmat)
