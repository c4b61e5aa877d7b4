"""Blocked Householder QR at the edges of the panel forms: one workgroup up to
1280 rows (forms of 128, 256, 512, 1024 and 1280 rows), workgroups of 512 rows
that exchange their sums beyond (1281: 3, 4097: 9, more than the 8 slots a
reader polls at once), and panels with fewer rows than columns."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
dp = C.POINTER(C.c_double)
NB = 32
EPS = np.finfo(float).eps


def d(a):
    return a.ctypes.data_as(dp)


@pytest.mark.parametrize("m,k", [(1, 3), (8, 8), (31, 40), (32, 32), (33, 32), (127, 33), (128, 31), (129, 65),
                                 (256, 32), (257, 20), (512, 33), (513, 7), (1024, 40), (1025, 33), (1280, 32),
                                 (1281, 32), (1313, 70), (2047, 33), (2600, 64), (4097, 33)])
def test_panel_forms(ktest, oracle, m, k):
    ktest.ktest_qr.argtypes = [C.c_int, C.c_int, dp, dp, dp, C.c_int, dp]
    rng = np.random.default_rng(m + 7 * k)
    A = np.asfortranarray(rng.standard_normal((m, k)) * np.logspace(0, -3, k))
    if k > 2:
        A[:, 1] = 0.0                      # tau = 0
        A[:, k - 1] = A[:, 0]              # a column that vanishes to rounding
    kk, nblk = min(m, k), (k + NB - 1) // NB
    P, tau, Tb = A.copy(order="F"), np.zeros(k), np.zeros((NB, NB * nblk), order="F")
    Cm = np.asfortranarray(rng.standard_normal((m, 5)))
    C2 = Cm.copy(order="F")
    assert ktest.ktest_qr(m, k, d(P), d(tau), d(Tb), 5, d(C2)) == 0
    V = np.tril(P[:, :kk], -1) + np.eye(m, kk)
    # the reflectors map A to R, and C to the updated C: errors of k
    # Householder steps, a small multiple of k eps in norm
    for M, got in ((A, np.triu(P[:kk])), (Cm, C2)):
        X = M.copy()
        for i in range(kk):
            X -= np.outer(tau[i] * V[:, i], V[:, i] @ X)
        want = X[:kk] if M is A else X
        assert np.linalg.norm(got - (np.triu(want) if M is A else want)) <= 20 * kk * EPS * np.linalg.norm(M)
        if M is A:
            assert np.linalg.norm(np.tril(X, -1)) <= 20 * kk * EPS * np.linalg.norm(M)
    # each is an orthogonal reflector with dlarfg's sign
    for i in range(kk):
        assert abs(tau[i] * (V[:, i] @ V[:, i]) - (2.0 if tau[i] else 0.0)) <= 100 * EPS
