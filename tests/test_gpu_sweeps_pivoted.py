"""The sweeps of LDL^T and LU at the edges of their kernels: fronts of at most 64 columns (one
workgroup, 256 rows below at a time, four columns of a wave together) with 0, 1, 255, 256, 257 and
2,047 - w rows below, fronts past those in 64-column steps, and right-hand sides around the groups of
one, two and four. A right-hand side goes through the same operations whichever others it is solved
with, so each column is compared bitwise with its solve alone; that solve's residual with the bound
of a triangular factorization, 3 n u |L| |U| |x| (src/solve/sweeps.jl:438-570).
"""
import numpy as np
import pytest
import scipy.sparse as sp

import sparsedirectsolver as sds
from sparsedirectsolver import matrices as M

pytestmark = pytest.mark.gpu


def _arrow(w, m, tail, symmetric):
    """w columns dense over themselves and m rows of a tail that is banded: a front of w columns with
    m rows below it, and the tail's own fronts. Strictly dominant, so that elements grow at most twofold."""
    rng = np.random.default_rng([w, m, tail, symmetric])
    n = w + max(m, tail)
    A = sp.lil_matrix((n, n))
    A[:w, :w] = rng.uniform(-1, 1, (w, w))
    rows = w + np.sort(rng.choice(n - w, m, replace=False))
    A[rows[:, None], np.arange(w)[None, :]] = rng.uniform(-1, 1, (m, w))
    A[np.arange(w)[:, None], rows[None, :]] = rng.uniform(-1, 1, (w, m))
    A = A.tocsr() + sp.diags(rng.uniform(-1, 1, n - 1), 1) + sp.diags(rng.uniform(-1, 1, n - 1), -1)
    if symmetric:
        A = sp.tril(A) + sp.tril(A, -1).T
    A = A - sp.diags(A.diagonal())
    sign = np.where(np.arange(n) % 3 == 0, -1.0, 1.0)
    return (A + sp.diags(sign * (1.0 + np.asarray(abs(A).sum(axis=0)).ravel()
                                 + np.asarray(abs(A).sum(axis=1)).ravel()))).tocsr()


@pytest.mark.parametrize("structure,view", [("S", "L"), ("G", "F")])
@pytest.mark.parametrize("w,m,tail,fp", [(1, 1, 5, "Float64"), (2, 0, 3, "Float64"), (15, 255, 300, "Float64"),
                                         (16, 256, 300, "Float32"), (17, 257, 300, "Float64"),
                                         (63, 64, 70, "Float32"), (64, 65, 70, "Float64"), (64, 1983, 1990, "Float64"),
                                         (65, 300, 310, "Float64"), (130, 300, 310, "Float32")])
def test_each_right_hand_side_as_alone(structure, view, w, m, tail, fp):
    import torch
    A = _arrow(w, m, tail, structure == "S")
    n = A.shape[0]
    A.sort_indices()
    rp, cv, nz = M.csr_arrays(M.lower_csr(A) if view == "L" else A)
    s = sds.DirectSolver((rp, cv, nz, n), structure, view)
    sds.setparam(s, "user_perm", np.arange(1, n + 1))
    sds.setparam(s, "amalgamation", (128, 0.25, 8))
    sds.setparam(s, "factor_precision", fp)
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    print(structure, w, m, fp, flush=True)
    B = np.random.default_rng(n).standard_normal((n, 64))
    dev = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    alone = np.zeros_like(B)
    modes = (0, 1) if structure == "G" else (0,)
    u = 2.0 ** -53 if fp == "Float64" else 2.0 ** -24
    for mode in modes:
        sds.setparam(s, "solve_mode", mode)
        for r in range(10):
            X = torch.zeros(n, dtype=torch.float64, device="cuda")
            sds.execute("solve", s, X, dev(B[:, r]))
            alone[:, r] = X.cpu().numpy()
        op = A.T if mode else A
        bound = 3.0 * n * u * 2.0 * abs(A).max() * np.abs(alone[:, :10]).sum(axis=0)
        assert (np.abs(op @ alone[:, :10] - B[:, :10]).max(axis=0) <= bound).all()
        for nrhs in (2, 3, 4, 5, 8, 9, 64):
            X = torch.zeros((n, nrhs), dtype=torch.float64, device="cuda")
            sds.execute("solve", s, X, dev(B[:, :nrhs]))
            k = min(nrhs, 10)
            assert np.array_equal(X.cpu().numpy()[:, :k], alone[:, :k]), nrhs
