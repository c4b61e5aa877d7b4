"""The blocked truncated pivoted QR where its kernels take other branches: columns
that a wave's registers do not hold during the selection (N beyond 3072, 4096
and 8192 for panels of two, four and eight waves), matrices whose squares leave
the range of the unscaled reflector scalars, and columns that are not finite."""
import numpy as np
import pytest

from test_gpu_rrqr import EPS, graded, q_apply, run

pytestmark = pytest.mark.gpu


def check(ktest, oracle, Cmat, tol, nd=1):
    k, N = Cmat.shape
    oracle.set_backend("own")
    Rref, jpvt, _ = oracle.geqp3(np.asfortranarray(Cmat))
    rank_ref = oracle.choose_rank(np.diag(Rref)[:min(k, N)], tol)
    rank, R, V, tau, perm, _ = run(ktest, Cmat, tol, nd=nd)
    assert rank == rank_ref
    assert np.array_equal(perm, jpvt[:rank])
    # backward error of r Householder steps: a small multiple of r eps |C|
    bar = 20 * max(rank, 1) * EPS * np.linalg.norm(Cmat)
    want = q_apply(V, tau, Cmat)[:rank]
    for p, j in enumerate(perm):
        want[p + 1:, j] = 0.0
    assert np.linalg.norm(R - want) <= bar


@pytest.mark.parametrize("k,N", [(49, 3100), (100, 4100), (200, 8300)])
def test_selection_beyond_registers(ktest, oracle, k, N):
    check(ktest, oracle, graded(k, N, 3, k + N), 1e-1)


# (n2 = alpha^2 + |x|^2 beyond 1e280, or below 1e-280 at the first pivots)
@pytest.mark.parametrize("nd", [1, 1000])
@pytest.mark.parametrize("scale", [1e145, 1e-145])
@pytest.mark.parametrize("k,N", [(30, 200), (100, 300)])
def test_scaled_reflectors(ktest, oracle, k, N, scale, nd):
    check(ktest, oracle, graded(k, N, 4, k) * scale, 1e-2, nd if k <= 48 else 1)


@pytest.mark.parametrize("nd", [1, 1000])
@pytest.mark.parametrize("k,N", [(30, 200), (48, 2100), (100, 300)])
def test_nan_columns(ktest, k, N, nd):
    """They are never pivots while another column is left: the rest is what it
    is beside columns of zeros."""
    Cmat = graded(k, N, 4, k)
    bad = [0, 17, N - 1]
    Cmat[:, bad] = 0.0
    want = run(ktest, Cmat, 1e-2, nd=nd if k <= 48 else 1)
    Cmat[3, bad] = np.nan
    got = run(ktest, Cmat, 1e-2, nd=nd if k <= 48 else 1)
    good = np.setdiff1d(np.arange(N), bad)
    assert got[0] == want[0] > 1
    assert np.array_equal(got[1][:, good], want[1][:, good])
    for a, b in zip(got[2:5], want[2:5]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_not_finite_first_pivot(ktest, value):
    """|r_00| is no number, so the test of the next step ends it: rank 1, as the
    column-by-column forms and the rule !(|r_11| / |r_00| >= tol) give it."""
    Cmat = graded(30, 200, 4, 30)
    if np.isnan(value):
        Cmat[:] = value
    else:
        Cmat[3, 7] = value
    rank, R, V, tau, perm, _ = run(ktest, Cmat, 1e-2)
    assert rank == 1 and perm[0] == (0 if np.isnan(value) else 7)
