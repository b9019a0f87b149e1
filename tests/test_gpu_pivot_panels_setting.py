"""The pivot-panel setting of a saved tuning keeps its meaning: 1 = panels (the default), 0 = one pivot per launch
pair, which holds no panel scratch."""
import numpy as np
import pytest

import sparsedirectsolver as sds

pytestmark = pytest.mark.gpu

TILES = dict(extend_add_rows=1024, cb_k_chunk=32, trailing_split=0, step_two_per_cu=0)


@pytest.mark.parametrize("structure,view", [("S", "L"), ("G", "F")])
def test_setting_selects_the_form(structure, view):
    n = 200
    A = np.random.default_rng(n).standard_normal((n, n))
    A = A + A.T
    if view == "L":
        cols = np.concatenate([np.arange(1, i + 2) for i in range(n)])
        rowptr, values = 1 + np.concatenate([[0], np.cumsum(np.arange(1, n + 1))]), A[np.tril_indices(n)]
    else:
        cols, rowptr, values = np.tile(np.arange(1, n + 1), n), 1 + n * np.arange(n + 1), A.reshape(-1)
    s = sds.DirectSolver((rowptr, cols, values, n), structure, view)
    sds.execute("analysis", s)
    sds.execute("factorization", s)

    def scratch():
        est = np.asarray(sds.getparam(s, "memory_estimates"))
        return est[1] - est[0] - est[8]

    default = scratch()
    assert default > 0
    for tiles, expected in ((dict(TILES, pivot_panels=0), 0), (dict(TILES, pivot_panels=1), default), (TILES, default)):
        sds.set_tiles(s, tiles)
        assert scratch() == expected, tiles
    assert sds.autotune(s, reps=1)["pivot_panels"] == 1
