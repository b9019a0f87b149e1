"""The solutions of a whole uniform batch go back to X in one strided copy: for every layout of X, also
one that is a view with strides of its own, they are those of the members solved one at a time
(ubatch_index), whose copies go member by member."""
import numpy as np
import pytest

import sparsedirectsolver as sds
from sparsedirectsolver import matrices as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["vector", "strided vector", "matrix", "transposed matrix", "array", "permuted array"])
@pytest.mark.parametrize("r", [1, 3])
def test_whole_batch_as_member_by_member(layout, r):
    import torch
    nb, dims = 4, (7, 6)
    mats = [M.lower_csr(M.variable_laplacian(dims, seed=k)) for k in range(nb)]
    rp, cv, _ = M.csr_arrays(mats[0])
    n = mats[0].shape[0]
    dev = dict(dtype=torch.float64, device="cuda")
    s = sds.DirectSolver((rp, cv, torch.tensor(np.concatenate([M.csr_arrays(A)[2] for A in mats]), **dev), n), "SPD", "L")
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    make = {"vector": lambda: torch.zeros(n * r * nb, **dev),
            "strided vector": lambda: torch.zeros(2 * n * r * nb, **dev)[::2],
            "matrix": lambda: torch.zeros((n, r * nb), **dev),
            "transposed matrix": lambda: torch.zeros((r * nb, n), **dev).t(),
            "array": lambda: torch.zeros((n, r, nb), **dev),
            "permuted array": lambda: torch.zeros((nb, n, r), **dev).permute(1, 2, 0)}[layout]
    X, Xk = make(), make()
    B = torch.tensor(np.random.default_rng(r).standard_normal(tuple(X.shape)), **dev)
    print(layout, r, flush=True)
    sds.execute("solve", s, X, B)
    for k in range(nb):
        sds.setparam(s, "ubatch_index", k)
        sds.execute("solve", s, Xk, B)
    assert torch.equal(X, Xk) and bool((X != 0).any())
