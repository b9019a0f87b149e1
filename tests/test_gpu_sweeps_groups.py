"""The Cholesky sweeps take right-hand sides in groups of 1, 2, 4 or 8 per workgroup, the grid's second
dimension covers them all (launch_rb): around every group size each column is bitwise its solve
alone, since a group gives each the same operations in the same order. The case has narrow fronts,
wide steps (more than 64 columns) with a narrow remainder, and fronts that finish their update vector in
the diagonal kernel.
"""
import numpy as np
import pytest

import sparsedirectsolver as sds
from sparsedirectsolver import matrices as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp", ["Float64", "Float32"])
@pytest.mark.parametrize("dims,amalgamation", [((13, 12, 11), (32, 0.25, 8)), ((17, 16, 15), (512, 0.25, 8))])
def test_each_right_hand_side_as_alone(dims, amalgamation, fp):
    import torch
    A = M.variable_laplacian(dims, seed=5)
    n = A.shape[0]
    rp, cv, nz = M.csr_arrays(M.lower_csr(A))
    s = sds.DirectSolver((rp, cv, nz, n), "SPD", "L")
    sds.setparam(s, "amalgamation", amalgamation)
    sds.setparam(s, "user_perm", sds.grid_nd_perm(*dims))
    sds.setparam(s, "factor_precision", fp)
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    print(dims, fp, flush=True)
    B = np.random.default_rng(n).standard_normal((n, 64))
    dev = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    alone = np.zeros((n, 18))
    for r in range(18):
        X = torch.zeros(n, dtype=torch.float64, device="cuda")
        sds.execute("solve", s, X, dev(B[:, r]))
        alone[:, r] = X.cpu().numpy()
    for nrhs in (2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 64):
        X = torch.zeros((n, nrhs), dtype=torch.float64, device="cuda")
        sds.execute("solve", s, X, dev(B[:, :nrhs]))
        k = min(nrhs, 18)
        assert np.array_equal(X.cpu().numpy()[:, :k], alone[:, :k]), nrhs
