"""LDL^T panels (pivot columns in registers) at the edges of their row classes, against one pivot per
launch pair: a dense symmetric matrix is one front whose remaining rows shrink through every panel
width. Both forms apply the reference's operations in the same order (src/reference/ldlt.jl:384-454),
so pivots, kinds, D, statistics and the panel are compared bitwise; no tolerance is involved.
"""
import numpy as np
import pytest

import sparsedirectsolver as sds
from sparsedirectsolver.solver import numeric_diag, numeric_factor, numeric_pivots, numeric_stats, set_tiles

pytestmark = pytest.mark.gpu

TILES = dict(extend_add_rows=1024, cb_k_chunk=32, trailing_split=0, step_two_per_cu=0)


# rows per thread change at 512; the panel widths at 3072, 5120 and 7168 rows (one pivot per launch
# pair above); a zero diagonal takes 2x2 pivots nearly everywhere (at panel ends too), a strong one
# mostly 1x1 pivots with interchanges now and then
@pytest.mark.parametrize("n,diag,ptype,fp", [(97, 0.0, "A", None), (513, 1.0, "A", None), (1041, 0.0, "B", None),
                                             (1300, 20.0, "D", None), (3080, 30.0, "A", None),
                                             (5130, 0.0, "A", None), (7190, 60.0, "A", None),
                                             (3090, 0.0, "A", "Float32")])
def test_panels_bitwise_as_one_pivot_per_launch(n, diag, ptype, fp):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A = A + A.T
    A[np.arange(n), np.arange(n)] = diag * rng.standard_normal(n)
    cols = np.concatenate([np.arange(1, i + 2) for i in range(n)])
    rowptr = 1 + np.concatenate([[0], np.cumsum(np.arange(1, n + 1))])
    s = sds.DirectSolver((rowptr, cols, A[np.tril_indices(n)], n), "S", "L")
    sds.setparam(s, "user_perm", np.arange(1, n + 1))
    sds.setparam(s, "pivot_pairs", "none")
    sds.setparam(s, "pivot_type", ptype)
    if fp:
        sds.setparam(s, "factor_precision", fp)
    sds.execute("analysis", s)
    assert s.symbolic.ns == 1
    print(f"n={n} diag={diag} {ptype} {fp or 'Float64'}", flush=True)
    out = []
    for pairs in (1, 0):
        set_tiles(s, dict(TILES, pivot_panels=pairs))
        sds.execute("factorization", s)
        out.append((numeric_pivots(s), numeric_diag(s), numeric_stats(s)[0], numeric_factor(s)))
    (p0, k0), d0, st0, f0 = out[0]
    (p1, k1), d1, st1, f1 = out[1]
    assert np.array_equal(p0, p1) and np.array_equal(k0, k1), "pivots differ"
    assert np.array_equal(d0, d1), "D differs"
    assert np.array_equal(st0, st1)
    assert np.array_equal(f0, f1)
