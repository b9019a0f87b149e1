"""LU panels (pivot columns in registers) at the edges of their row classes, against one pivot per
launch pair: a dense matrix is one front whose remaining rows shrink through every panel width, an
arrow matrix a front with rows below its columns and a wide U12. Both forms apply the reference's
operations in the same order (src/reference/lu.jl:163-214), so row order, D, statistics and both
panels are compared bitwise; no tolerance is involved.
"""
import numpy as np
import pytest

import sparsedirectsolver as sds
from sparsedirectsolver.solver import numeric_diag, numeric_factor, numeric_pivots, numeric_stats, set_tiles

pytestmark = pytest.mark.gpu

TILES = dict(extend_add_rows=1024, cb_k_chunk=32, trailing_split=0, step_two_per_cu=0)


def _both(s):
    out = []
    for pairs in (1, 0):
        set_tiles(s, dict(TILES, pivot_panels=pairs))
        sds.execute("factorization", s)
        out.append((numeric_pivots(s), numeric_diag(s), numeric_stats(s)[0], numeric_factor(s), numeric_factor(s, 1)))
    (p0, k0), d0, st0, l0, u0 = out[0]
    (p1, k1), d1, st1, l1, u1 = out[1]
    assert np.array_equal(p0, p1) and np.array_equal(k0, k1), "row order differs"
    assert np.array_equal(d0, d1), "D differs"
    assert np.array_equal(st0, st1)
    assert np.array_equal(l0, l1) and np.array_equal(u0, u1)
    return p0


# rows per thread change at 512; the panel widths at 1536, 3072, 5120 rows; threshold 1 interchanges
# nearly every row, a small one on a strong diagonal almost none; "N" never (with pivots below
# epsilon, perturbed)
@pytest.mark.parametrize("n,diag,threshold,ptype,fp", [(91, 0.0, 1.0, "A", None), (513, 4.0, 0.1, "A", None),
                                                       (530, 1.0, 0.5, "N", None), (1545, 0.0, 0.5, "A", None),
                                                       (3080, 60.0, 0.1, "A", None), (5130, 20.0, 0.2, "A", None),
                                                       (1545, 0.0, 1.0, "A", "Float32")])
def test_panels_bitwise_as_one_pivot_per_launch(n, diag, threshold, ptype, fp):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    A[np.arange(n), np.arange(n)] += diag * rng.standard_normal(n)
    if ptype == "N":
        A[0, 0] = 0.0
    rowptr = 1 + n * np.arange(n + 1)
    s = sds.DirectSolver((rowptr, np.tile(np.arange(1, n + 1), n), A.reshape(-1), n), "G", "F")
    sds.setparam(s, "user_perm", np.arange(1, n + 1))
    sds.setparam(s, "pivot_type", ptype)
    sds.setparam(s, "pivot_threshold", threshold)
    if fp:
        sds.setparam(s, "factor_precision", fp)
    sds.execute("analysis", s)
    assert s.symbolic.ns == 1
    print(f"n={n} diag={diag} u={threshold} {ptype} {fp or 'Float64'}", flush=True)
    piv = _both(s)
    if ptype == "A" and diag == 0.0:
        assert not np.array_equal(piv, np.arange(1, n + 1))


@pytest.mark.parametrize("w,m", [(1, 90), (8, 300), (33, 70), (40, 1600), (130, 131)])
def test_panels_with_rows_below(w, m):
    """w interior columns per leaf front coupled to a dense border of m rows (two leaves, one root)."""
    rng = np.random.default_rng(100 * w + m)
    n = 2 * w + m
    A = np.zeros((n, n))
    for b in range(2):
        i = slice(b * w, (b + 1) * w)
        A[i, i] = rng.standard_normal((w, w))
        A[i, 2 * w:] = rng.standard_normal((w, m))
        A[2 * w:, i] = rng.standard_normal((m, w))
    A[2 * w:, 2 * w:] = rng.standard_normal((m, m))
    rows, cols = np.nonzero(A)
    rowptr = 1 + np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    s = sds.DirectSolver((rowptr, cols + 1, A[rows, cols], n), "G", "F")
    sds.setparam(s, "user_perm", np.arange(1, n + 1))
    sds.setparam(s, "amalgamation", (4096, 0.0, 0))
    sds.setparam(s, "pivot_threshold", 0.5)
    sds.execute("analysis", s)
    print(f"w={w} m={m}: fronts {list(zip(s.symbolic.front_nrows, s.symbolic.front_ncols))[:4]}", flush=True)
    assert max(s.symbolic.front_nrows) == max(m, w + m)
    _both(s)
