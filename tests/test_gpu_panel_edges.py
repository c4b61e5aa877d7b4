"""The panel kernel where its own tests do not reach: FP32 panels at the edges of
their forms (2048 rows in one workgroup, the exchange beyond), squares outside the
range of the unscaled reflector scalars, a column that is not finite; and the
FP32 block T factors."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NB = 32


def kinds(f32):
    t = np.float32 if f32 else np.float64
    return t, C.POINTER(C.c_float if f32 else C.c_double), np.finfo(t).eps


def qr(ktest, f32, A, Cm):
    t, tp, _ = kinds(f32)
    f = ktest.ktest_qr_f32 if f32 else ktest.ktest_qr
    f.argtypes = [C.c_int, C.c_int, tp, tp, tp, C.c_int, tp]
    m, k = A.shape
    P, tau = np.array(A, dtype=t, order="F"), np.zeros(k, t)
    Tb, C2 = np.zeros((NB, NB * ((k + NB - 1) // NB)), t, order="F"), np.array(Cm, dtype=t, order="F")
    p = lambda M: M.ctypes.data_as(tp)
    assert f(m, k, p(P), p(tau), p(Tb), Cm.shape[1], p(C2)) == 0
    return P.astype(float), tau.astype(float), Tb.astype(float), C2.astype(float)


def check(ktest, f32, A, Cm):
    """A, Cm representable in the type."""
    m, k = A.shape
    eps, kk = kinds(f32)[2], min(m, k)
    P, tau, _, C2 = qr(ktest, f32, A, Cm)
    V = np.tril(P[:, :kk], -1) + np.eye(m, kk)
    # the reflectors map A to R, and C to the updated C: errors of k Householder
    # steps, a small multiple of k eps in norm
    for M, got in ((A, np.triu(P[:kk])), (Cm, C2)):
        X = M.copy()
        for i in range(kk):
            X -= np.outer(tau[i] * V[:, i], V[:, i] @ X)
        want = np.triu(X[:kk]) if M is A else X
        assert np.linalg.norm(got - want) <= 20 * kk * eps * np.linalg.norm(M)
        if M is A:
            assert np.linalg.norm(np.tril(X, -1)) <= 20 * kk * eps * np.linalg.norm(M)
    # orthogonal reflectors: |x|^2 is a sum of up to 32 terms a lane, then over 8
    # lanes, 8 waves and 9 workgroups, so tau v^T v = 2 to 2 (32 + 8 + 8 + 9 + 10) eps
    for i in range(kk):
        assert abs(tau[i] * (V[:, i] @ V[:, i]) - (2.0 if tau[i] else 0.0)) <= 150 * eps


def data(m, k, f32):
    rng = np.random.default_rng(m + 7 * k)
    t = kinds(f32)[0]
    A = rng.standard_normal((m, k)) * np.logspace(0, -3, k)
    if k > 2:
        A[:, 1] = 0.0  # tau = 0
    return A.astype(t).astype(float), rng.standard_normal((m, 5)).astype(t).astype(float)


@pytest.mark.parametrize("m,k", [(1, 3), (31, 40), (33, 32), (128, 33), (129, 65), (256, 20), (257, 33), (512, 7),
                                 (1025, 40), (1281, 32), (2047, 33), (2048, 33), (2049, 32), (2600, 64), (4097, 33)])
def test_panel_forms_f32(ktest, m, k):
    check(ktest, True, *data(m, k, True))


# alpha^2 + |x|^2 beyond 1e280 (1e30 in FP32) or below 1e-280 (1e-30)
@pytest.mark.parametrize("f32,scale", [(False, 1e145), (False, 1e-145), (True, 2.0**53), (True, 2.0**-56)])
@pytest.mark.parametrize("m,k", [(20, 33), (200, 40), (1000, 33), (2600, 20)])
def test_scaled_reflectors(ktest, f32, scale, m, k):
    rng = np.random.default_rng(m)
    t = kinds(f32)[0]
    A, Cm = (rng.standard_normal((m, n)).astype(t).astype(float) for n in (k, 5))
    check(ktest, f32, (A * scale).astype(t).astype(float), Cm)


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("m,k,j", [(40, 33, 5), (300, 40, 33), (2600, 20, 7)])
def test_not_finite_column(ktest, f32, m, k, j, value):
    """R's columns and the scalars before it are what they are without it, and
    the column shows that it is no number.  (The earlier reflectors' entries meet
    x times zero and are not kept; the block's T factor is no number either, so
    nothing that the block is applied to is.)"""
    A, Cm = data(m, k, f32)
    want = qr(ktest, f32, A, Cm)
    A[m - 1, j] = value
    got = qr(ktest, f32, A, Cm)
    assert np.array_equal(np.triu(got[0])[:j, :j], np.triu(want[0])[:j, :j])
    assert np.array_equal(got[1][:j], want[1][:j])
    assert not np.all(np.isfinite(got[0][:, j]))
    jb = j // NB * NB
    assert not np.all(np.isfinite(got[2][:, jb:jb + NB]))


@pytest.mark.parametrize("m,r", [(1, 1), (16, 16), (33, 17), (40, 33), (300, 64), (1000, 100)])
def test_larft_f32(ktest, m, r):
    f = ktest.ktest_larft_f32
    fp = C.POINTER(C.c_float)
    f.argtypes = [C.c_int, C.c_int, fp, fp, fp]
    rng = np.random.default_rng(m + r)
    V = np.asfortranarray(rng.standard_normal((m, r)).astype(np.float32) / np.float32(np.sqrt(m)))
    Vd = np.tril(V.astype(float), -1) + np.eye(m, r)
    tau = (2.0 / np.sum(Vd * Vd, axis=0)).astype(np.float32)
    nblk = (r + NB - 1) // NB
    Tb = np.full((NB, NB * nblk), np.nan, np.float32, order="F")
    p = lambda M: M.ctypes.data_as(fp)
    assert f(m, r, p(V), p(tau), p(Tb)) == 0
    eps = np.finfo(np.float32).eps
    for jb in range(0, r, NB):
        w = min(NB, r - jb)
        Vb = Vd[jb:, jb:jb + w]
        # T^{-1} = diag(1 / tau) + the strict upper part of V^T V
        G = np.triu(Vb.T @ Vb, 1)
        T = np.linalg.inv(np.diag(1.0 / tau[jb:jb + w].astype(float)) + G)
        # products of m - jb terms, then a recurrence of w steps on T
        n2 = np.linalg.norm(T, 2)
        bound = eps * ((m - jb + 2) * np.linalg.norm(abs(Vb).T @ abs(Vb)) * n2**2 + 64 * np.linalg.cond(T) * n2)
        got = Tb[:, jb:jb + NB].astype(float)
        assert np.linalg.norm(got[:w, :w] - T) <= bound
        assert not np.any(np.tril(got, -1)) and not np.any(got[:, w:])
