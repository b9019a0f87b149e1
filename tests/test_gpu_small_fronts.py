"""The kernels of the small Cholesky fronts at their edges: the one-wave kernel (at most 32 rows), the
blocked kernel with one or two rows a lane (at most 64 rows, more), panels of fewer than 16 columns,
enough fronts of at most 64 rows for a launch of their own, and a front with more than 64 children.
They apply the operations of the column-by-column kernel in its order (src/numeric/front.jl:154-206),
so the factors are compared bitwise, and a solve's residual with the standard bound of a Cholesky
solve.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import sparsedirectsolver as sds
from sparsedirectsolver import matrices as M
from sparsedirectsolver.solver import numeric_factor, set_tiles

pytestmark = pytest.mark.gpu

TILES = dict(extend_add_rows=1024, cb_k_chunk=32, trailing_split=0, step_two_per_cu=0)


def _spd(rng, n):
    a = rng.standard_normal((n, n))
    return a @ a.T + n * np.eye(n)


def _dense(sizes):
    rng = np.random.default_rng(list(sizes))
    return sp.block_diag([_spd(rng, n) for n in sizes], format="csr")


def _star(leaves, core):
    """`leaves` single columns, each tied to the same two and one other of `core` columns"""
    rng = np.random.default_rng([leaves, core])
    n = leaves + core
    A = np.zeros((n, n))
    A[leaves:, leaves:] = _spd(rng, core)
    for c in range(leaves):
        for r in (leaves, leaves + 1, leaves + 2 + c % (core - 2)):
            A[r, c] = A[c, r] = rng.standard_normal()
        A[c, c] = 3.0 * leaves
    A[np.arange(leaves, n), np.arange(leaves, n)] += leaves
    return sp.csr_matrix(A)


def _solve(s, b):
    import torch
    B = torch.tensor(b, dtype=torch.float64, device="cuda")
    X = torch.zeros_like(B)
    sds.execute("solve", s, X, B)
    return X.cpu().numpy()


CASES = [("chains", lambda: _dense([1, 2, 15, 16, 17, 31, 32, 33, 47, 63, 64, 65, 79, 80, 81, 89, 90]), (32, 0.25, 8)),
         ("whole", lambda: _dense([31, 32, 33, 48, 63, 64, 65, 79, 80, 90]), (512, 0.25, 8)),
         ("many_low", lambda: _dense([40] * 515 + [70] * 3), (512, 0.25, 8)),
         ("star_tiny", lambda: _star(70, 20), (32, 0.0, 1)),
         ("star_mid", lambda: _star(131, 45), (32, 0.0, 1))]


@pytest.mark.parametrize("fp", ["Float64", "Float32"])
@pytest.mark.parametrize("name,make,amalgamation", CASES, ids=[c[0] for c in CASES])
def test_small_fronts(name, make, amalgamation, fp):
    A = make()
    n = A.shape[0]
    rp, cv, nz = M.csr_arrays(M.lower_csr(A))
    s = sds.DirectSolver((rp, cv, nz, n), "SPD", "L")
    sds.setparam(s, "amalgamation", amalgamation)
    sds.setparam(s, "user_perm", np.arange(1, n + 1))
    sds.setparam(s, "factor_precision", fp)
    sds.execute("analysis", s)
    if name.startswith("star"):
        assert np.diff(s.symbolic.maps["child_ptr"]).max() > 64
    print(name, fp, flush=True)
    factors = []
    for kind in (2, 0):
        set_tiles(s, dict(TILES, small_front_kernel=kind))
        sds.execute("factorization", s)
        assert sds.getparam(s, "info") == 0
        factors.append(numeric_factor(s))
    assert np.array_equal(factors[0], factors[1])
    # |b - A x| <= gamma_{3 k + 1} |L| |L^T| |x|, k the longest row of L (a block); an entry of
    # |L| |L^T| is at most max a_ii by Cauchy-Schwarz, and a row has at most n of them
    u = 2.0 ** -53 if fp == "Float64" else 2.0 ** -24
    B = np.random.default_rng(n).standard_normal(n)
    X = _solve(s, B)
    k = n if name.startswith("star") else max(np.diff(A.indptr))
    bound = (3.0 * k + 2.0) * u * A.diagonal().max() * n * np.abs(X).max()
    assert np.abs(A @ X - B).max() <= bound


@pytest.mark.parametrize("n,bad", [(20, 0), (20, 7), (20, 19), (60, 0), (60, 16), (60, 41), (85, 33), (85, 84)])
def test_a_failed_pivot_is_reported_at_its_column(n, bad):
    """a matrix that is positive definite up to column `bad`: every kernel reports that column, and
    after the values are mended the factor is that of the mended matrix"""
    A = _spd(np.random.default_rng(n), n)
    rp, cv, good = M.csr_arrays(M.lower_csr(sp.csr_matrix(A)))
    nz = np.array(good)
    nz[(np.cumsum(np.arange(1, n + 1)) - 1)[bad]] = -1.0
    s = sds.DirectSolver((rp, cv, nz, n), "SPD", "L")
    sds.setparam(s, "amalgamation", (512, 0.25, 8))
    sds.setparam(s, "user_perm", np.arange(1, n + 1))
    sds.execute("analysis", s)
    assert s.symbolic.ns == 1
    for kind in (2, 0):
        set_tiles(s, dict(TILES, small_front_kernel=kind))
        sds.execute("factorization", s)
        assert sds.getparam(s, "info") == bad + 1
    sds.update(s, good)
    factors = []
    for kind in (2, 0):
        set_tiles(s, dict(TILES, small_front_kernel=kind))
        sds.execute("factorization", s)
        assert sds.getparam(s, "info") == 0
        factors.append(numeric_factor(s))
    assert np.array_equal(factors[0], factors[1])
