"""The block update of a Householder step, C <- (I - V T V^T)^T C, in one kernel:
every form at its largest number of rows, one less and one more than the form
before holds, partial row tiles, partial reflector blocks, several targets."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
dp, fp = C.POINTER(C.c_double), C.POINTER(C.c_float)
FORM_ROWS = [64, 128, 256, 384, 512, 768, 1024, 1536, 2048]
CASES = [(0, 1, 1, 1), (0, 5, 16, 5), (0, 33, 17, 32), (1, 17, 3, 16), (2, 64, 40, 17), (8, 40, 33, 31)]
CASES += [(f, r, 20 + f, w) for f, top in enumerate(FORM_ROWS)
          for r, w in ((top, 32), (top - 1, 32), (top // 2 + 18, 19))]


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("form,rows,cols,w", CASES)
def test_larfb(ktest, f32, form, rows, cols, w):
    assert ktest.ktest_larfb_rows(form) == FORM_ROWS[form]
    rng = np.random.default_rng(rows + 3 * w + form)
    t, tp, f = (np.float32, fp, ktest.ktest_larfb_f32) if f32 else (np.float64, dp, ktest.ktest_larfb)
    i = C.c_int
    f.argtypes = [i, i, i, i, i, tp, i, tp, tp, i]
    eps, nt, ldv, ldc = np.finfo(t).eps, 3, rows + 3, rows + 1
    V = np.full((ldv, w), np.nan, t, order="F")   # R lies above the diagonal, other data below
    V[:rows] = rng.standard_normal((rows, w)) / np.sqrt(rows)
    V[:rows][np.triu_indices(rows, 0, w)] = np.nan
    Tb = np.zeros((32, 32), t, order="F")
    Tb[:w, :w] = np.triu(rng.standard_normal((w, w)))
    Cm = np.full((ldc, nt * cols), 7.0, t, order="F")
    Cm[:rows] = rng.standard_normal((rows, nt * cols))
    Vd = np.where(np.tri(rows, w, -1) > 0, V[:rows], 0).astype(float) + np.eye(rows, w)
    Td, Cd = Tb[:w, :w].astype(float), Cm[:rows].astype(float)
    want = Cd - Vd @ (Td.T @ (Vd.T @ Cd))
    got = Cm.copy(order="F")
    p = lambda M: M.ctypes.data_as(tp)
    assert f(form, rows, cols, nt, w, p(V), ldv, p(Tb), p(got), ldc) == 0
    # three products of rows, w and w terms
    bound = (rows + 2 * w + 4) * eps * (abs(Cd) + abs(Vd) @ (abs(Td).T @ (abs(Vd).T @ abs(Cd))))
    assert np.all(abs(got[:rows] - want) <= bound)
    assert np.all(got[rows:] == 7.0)
