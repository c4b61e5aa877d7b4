"""Device memory that closed trees leave for the next ones goes back on request."""
import numpy as np
import pytest

import spaqr_public_amd as sq
from spaqr_public_amd import gen

pytestmark = pytest.mark.gpu


def test_pool_trim():
    import torch
    A, _ = sq.colscale(gen.config_matrix("advdiff2d_64"))
    b = np.random.default_rng(0).standard_normal(A.shape[0])

    def tree():
        t = sq.Tree(sq.default_levels(A.shape[1]), 0, sq.FP64)
        t.set_scale(1)
        t.set_tol(1e-3)
        t.set_square(1)
        t.set_tensor_coordinates(64, 2)
        t.partition(A)
        t.assemble(A)
        t.factorize()
        return t

    alive = tree()
    x = alive.solve(b)
    other = tree()
    held = other.counters()["device_bytes"]
    other.close()
    before = torch.cuda.mem_get_info()[0]
    sq.pool_trim()
    assert torch.cuda.mem_get_info()[0] - before >= held > 0
    assert np.array_equal(alive.solve(b), x)  # what a tree uses stays
    again = tree()
    assert np.array_equal(again.solve(b), x)
    alive.close()
    again.close()
