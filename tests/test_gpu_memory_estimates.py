"""The memory estimates count the pivot panels' scratch (src/symbolic/maps.jl:338-356 counts what the numeric phase
holds)."""
import numpy as np
import pytest

import sparsedirectsolver as sds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("structure,view", [("S", "L"), ("G", "F")])
def test_estimates_hold_the_panel_scratch(structure, view):
    n = 300
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A = A + A.T
    if view == "L":
        cols = np.concatenate([np.arange(1, i + 2) for i in range(n)])
        rowptr, values = 1 + np.concatenate([[0], np.cumsum(np.arange(1, n + 1))]), A[np.tril_indices(n)]
    else:
        cols, rowptr, values = np.tile(np.arange(1, n + 1), n), 1 + n * np.arange(n + 1), A.reshape(-1)
    s = sds.DirectSolver((rowptr, cols, values, n), structure, view)
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    est = np.asarray(sds.getparam(s, "memory_estimates"))
    assert est[1] >= est[0] + est[8] + 8 * 16 * n  # a panel of 16 columns or more of the one front
