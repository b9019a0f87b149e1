"""Pivot panels against one pivot per launch pair in the register classes and row slots that the dense fronts of
test_gpu_ldlt_panels.py and test_gpu_lu_panels.py leave out: LDL^T with 3 rows a thread up to its edge, the 8- and
4-column classes in FP32, LU with every one of the 4-column class's 20
row slots and all classes in FP32. Both forms apply the reference's
operations in the same order (src/reference/ldlt.jl:384-454, lu.jl:163-214): compared bitwise.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import sparsedirectsolver as sds
from sparsedirectsolver.solver import numeric_diag, numeric_factor, numeric_pivots, numeric_stats, set_tiles

pytestmark = pytest.mark.gpu

TILES = dict(extend_add_rows=1024, cb_k_chunk=32, trailing_split=0, step_two_per_cu=0)


def _both(s, sides):
    out = []
    for form in (0, 1):
        set_tiles(s, dict(TILES, pivot_panels=form))
        sds.execute("factorization", s)
        out.append((*numeric_pivots(s), numeric_diag(s), numeric_stats(s)[0], *(numeric_factor(s, q) for q in sides)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# 1,545 rows: 3 rows a thread from 1,536 on; FP32: 5,130 rows the 8-column class, 7,190 the 4-column one
@pytest.mark.parametrize("n,diag,ptype,fp", [(1545, 1.0, "A", None), (1545, 0.0, "D", "Float32"),
                                             (5130, 1.0, "A", "Float32"), (7190, 40.0, "A", "Float32")])
def test_ldlt_classes(n, diag, ptype, fp):
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
    _both(s, (0,))


# one front of w + m rows (w full rows and columns, a border of m): all 20 slots of the 4-column class, the
# last one partly filled, then every other class as the rows grow fewer
@pytest.mark.parametrize("w,m,fp", [(24, 10210, None), (24, 10210, "Float32")])
def test_lu_classes(w, m, fp):
    rng = np.random.default_rng(w + m)
    A = sp.bmat([[rng.standard_normal((w, w)), rng.standard_normal((w, m))],
                 [rng.standard_normal((m, w)), sp.diags(10.0 * rng.standard_normal(m))]]).tocsr()
    A.sort_indices()
    n = w + m
    s = sds.DirectSolver((A.indptr + 1, A.indices + 1, A.data, n), "G", "F")
    sds.setparam(s, "user_perm", np.arange(1, n + 1))
    sds.setparam(s, "amalgamation", (1, 0.0, 0))
    sds.setparam(s, "pivot_threshold", 0.5)
    if fp:
        sds.setparam(s, "factor_precision", fp)
    sds.execute("analysis", s)
    print(f"w={w} m={m} {fp or 'Float64'}: fronts {list(zip(s.symbolic.front_nrows, s.symbolic.front_ncols))[:4]}",
          flush=True)
    assert max(s.symbolic.front_nrows) == n
    _both(s, (0, 1))
