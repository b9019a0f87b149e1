"""The work a user of this solver has it do, as timed cases.

A program analyses a matrix pattern once and then runs the numeric phase again and again: a
refactorization with new values, solves with it, gradients through it. Each case is one such pass
through the public entry points of the Python package (DirectSolver / execute / getparam,
UnevenBatch, graph_capture / graph_replay, SparseSolve). The matrices are the families of
bench.py and the tests: variable-coefficient Laplacians on 2-D and 3-D grids (SPD), the KKT
generator (symmetric indefinite), upwind convection-diffusion (unsymmetric).

Analysis, buffers and the first factorization belong to ``prepare``; a pass is what the program
repeats.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sparsedirectsolver.jl_amd"))

import sparsedirectsolver as sds  # noqa: E402
from sparsedirectsolver import matrices as M  # noqa: E402
from sparsedirectsolver.adjoint import SparseSolve  # noqa: E402
from sparsedirectsolver.batch import UnevenBatch  # noqa: E402
from sparsedirectsolver.solver import graph_capture, graph_replay  # noqa: E402


def listed():
    return [
        # a small 2-D mesh problem solved per time step: the smallest calls, latency and launches count
        dict(name="spd 2d 31x29", kind="spd", dims="31x29", fp="Float64", nrhs=1, ir=0, wide=False, op="step"),
        # an ordinary 3-D diffusion problem at the package's default options, odd sizes
        dict(name="spd 3d 27x26x23", kind="spd", dims="27x26x23", fp="Float64", nrhs=1, ir=0, wide=False, op="step"),
        # the benchmark workload: 64^3, 8 right-hand sides, wide supernodes, Float64
        dict(name="spd 3d 64 8rhs", kind="spd", dims="64x64x64", fp="Float64", nrhs=8, ir=0, wide=True, op="step"),
        # a Float32 factor with Float64 refinement
        dict(name="spd 3d 47 f32+ir", kind="spd", dims="47x47x47", fp="Float32", nrhs=1, ir=2, wide=True, op="step"),
        # many right-hand sides on a factor in hand (modal analysis, load cases): solve only
        dict(name="spd 3d 40 solve 24rhs", kind="spd", dims="40x40x40", fp="Float64", nrhs=24, ir=0, wide=False,
             op="solve"),
        # interior-point steps: refactorization, the inertia, a refined solve; small, ordinary, large
        dict(name="kkt 1500 f32 fgmres", kind="kkt", nh=1000, fp="Float32", mode="fgmres", ir=6, wide=False),
        dict(name="kkt 4521", kind="kkt", nh=3014, fp="Float64", mode="ir", ir=2, wide=False),
        dict(name="kkt 12000", kind="kkt", nh=8000, fp="Float64", mode="ir", ir=2, wide=True),
        # unsymmetric transport: a step with badly scaled rows (row interchanges), a transposed solve too
        dict(name="lu 3d 19 rows scaled", kind="lu", k=19, fp="Float64", nrhs=3, wide=False, scaled=True, op="step"),
        # differentiation through the solver: refactorization, solve, gradients of values and right-hand side
        dict(name="lu 3d 32 gradient", kind="lu", k=32, fp="Float64", nrhs=1, wide=True, scaled=False, op="gradient"),
        # many small systems of one pattern, and of different sizes from one graph
        dict(name="uniform batch 96", kind="uniform", members=96, nx=23, ny=18, nrhs=2, fp="Float64"),
        dict(name="uneven batch 160 f32+ir", kind="uneven", members=160, lo=24, hi=140, fp="Float32", ir=1),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["spd2", "spd3", "spd3", "solve", "kkt", "kkt", "lu", "lu", "uniform", "uneven"])
    fp = rng.choice(["Float64", "Float64", "Float32"])
    ir = 0 if fp == "Float64" else 2
    wide = rng.random() < 0.5
    if kind == "spd2":
        dims = "%dx%d" % (_log(rng, 20, 400), _log(rng, 20, 400))
        return dict(kind="spd", dims=dims, fp=fp, nrhs=rng.choice([1, 2, 5]), ir=ir, wide=wide, op="step")
    if kind == "spd3":
        k = _log(rng, 12, 56)
        dims = "%dx%dx%d" % (k, max(3, k - rng.randrange(4)), max(3, k + rng.randrange(-3, 3)))
        return dict(kind="spd", dims=dims, fp=fp, nrhs=rng.choice([1, 3, 8]), ir=ir, wide=wide, op="step")
    if kind == "solve":
        k = _log(rng, 12, 44)
        dims = "%dx%dx%d" % (k, k + 1, max(3, k - rng.randrange(3)))
        return dict(kind="spd", dims=dims, fp="Float64", nrhs=_log(rng, 1, 64), ir=0, wide=wide, op="solve")
    if kind == "kkt":
        nh = _log(rng, 500, 7000)
        return dict(kind="kkt", nh=nh, fp=fp, mode="ir" if fp == "Float64" else "fgmres",
                    ir=2 if fp == "Float64" else 6, wide=wide)
    if kind == "lu":
        k = _log(rng, 8, 30)
        if rng.random() < 0.4:
            return dict(kind="lu", k=k, fp="Float64", nrhs=1, wide=wide, scaled=False, op="gradient")
        return dict(kind="lu", k=k, fp="Float64", nrhs=rng.choice([1, 3, 7]), wide=wide, scaled=rng.random() < 0.5,
                    op="step")
    if kind == "uniform":
        return dict(kind="uniform", members=_log(rng, 8, 128), nx=rng.randrange(9, 40), ny=rng.randrange(9, 40),
                    nrhs=rng.choice([1, 2]), fp="Float64")
    return dict(kind="uneven", members=_log(rng, 16, 160), lo=24, hi=rng.randrange(60, 141), fp="Float32", ir=1)


# -- matrices: the pattern of a case, values by the seed -----------------------------------------------

def _dims(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _kkt(case, seed):
    """The generator's pattern (always the same one for a size, as along the steps of an interior-point
    method), its Hessian block with a barrier diagonal and its variables in units of the seed's:
    D (K + [Sigma 0; 0 0]) D, whose inertia is K's."""
    nh, nj = case["nh"], case["nh"] // 2
    K = M.kkt_matrix(nh, nj)
    rng = np.random.default_rng([3, seed])
    d = np.exp(0.3 * rng.standard_normal(nh + nj))
    sigma = np.concatenate([10.0 ** rng.uniform(-2.0, 1.0, nh), np.zeros(nj)])
    rows = np.repeat(np.arange(nh + nj), np.diff(K.indptr))
    data = K.data + np.where(rows == K.indices, sigma[rows], 0.0)
    K.data = d[rows] * data * d[K.indices]
    return K


def _lu(case, seed):
    A = M.convection_diffusion3d(case["k"], peclet=10.0).tocsr()
    A.sort_indices()
    rng = np.random.default_rng([7, seed])
    A.data = A.data * (1.0 + 0.1 * rng.uniform(-1.0, 1.0, A.data.size))
    if case["scaled"]:  # equations in units of their own
        r = 10.0 ** rng.uniform(-2.0, 2.0, A.shape[0])
        A.data = A.data * np.repeat(r, np.diff(A.indptr))
    return A


def _members(case, seed):
    """sides of an uneven batch: the sizes are the case's, the coefficients the seed's"""
    sides = np.exp(np.random.default_rng(case["members"]).uniform(np.log(case["lo"]), np.log(case["hi"] + 0.5),
                                                                  case["members"]))
    return [(int(q), M.variable_laplacian((int(q), int(q)), seed=[seed, j])) for j, q in enumerate(sides)]


def _uniform(case, seed):
    return [M.variable_laplacian((case["nx"], case["ny"]), seed=[seed, j]) for j in range(case["members"])]


def _normal(seed, stream, *shape):
    return np.random.default_rng([stream, seed]).standard_normal(shape)


def _device(a):
    return torch.tensor(a, dtype=torch.float64, device="cuda")


def _options(s, case):
    sds.setparam(s, "factor_precision", case["fp"])
    if case.get("wide"):  # wide supernodes, as the benchmark sets them
        sds.setparam(s, "amalgamation", (512, 0.25, 8))


# -- prepare and run -------------------------------------------------------------------------------------

def prepare(case, seed):
    return {"spd": _prepare_spd, "kkt": _prepare_kkt, "lu": _prepare_lu, "uniform": _prepare_uniform,
            "uneven": _prepare_uneven}[case["kind"]](case, seed)


def _prepare_spd(case, seed):
    A = M.variable_laplacian(_dims(case), seed=seed)
    rp, cv, nz = M.csr_arrays(M.lower_csr(A))
    n = A.shape[0]
    s = sds.DirectSolver((rp, cv, _device(nz), n), "SPD", "L")
    _options(s, case)
    if case["wide"]:
        sds.setparam(s, "reordering_alg", "algo4")
    sds.setparam(s, "ir_n_steps", case["ir"])
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    B = _device(_normal(seed, 1, n, case["nrhs"]))
    return dict(case=case, solver=s, B=B, X=torch.zeros_like(B))


def _prepare_kkt(case, seed):
    K = _kkt(case, seed)
    rp, cv, nz = M.csr_arrays(M.lower_csr(K))
    n = K.shape[0]
    s = sds.DirectSolver((rp, cv, _device(nz), n), "S", "L")
    _options(s, case)
    sds.setparam(s, "reordering_alg", "algo3")
    sds.setparam(s, "ir_mode", case["mode"])
    sds.setparam(s, "ir_n_steps", case["ir"])
    if case["mode"] == "fgmres":
        sds.setparam(s, "ir_tol", 1e-14)
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    B = _device(_normal(seed, 1, n))
    return dict(case=case, solver=s, B=B, X=torch.zeros_like(B))


def _prepare_lu(case, seed):
    A = _lu(case, seed)
    rp, cv, nz = M.csr_arrays(A)
    n = A.shape[0]
    values = _device(nz)
    s = sds.DirectSolver((rp, cv, values, n), "G", "F")
    _options(s, case)
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    if case["op"] == "gradient":
        b = _device(_normal(seed, 1, n))
        return dict(case=case, solver=s, values=values.requires_grad_(), b=b.requires_grad_(),
                    xbar=_device(_normal(seed, 2, n)))
    B = _device(_normal(seed, 1, n, case["nrhs"]))
    return dict(case=case, solver=s, B=B, X=torch.zeros_like(B), Xt=torch.zeros_like(B))


def _prepare_uniform(case, seed):
    mats = [M.lower_csr(A) for A in _uniform(case, seed)]
    rp, cv, _ = M.csr_arrays(mats[0])
    n, nb = mats[0].shape[0], case["members"]
    values = _device(np.concatenate([M.csr_arrays(A)[2] for A in mats]))
    s = sds.DirectSolver((rp, cv, values, n), "SPD", "L")
    _options(s, case)
    sds.execute("analysis", s)
    sds.execute("factorization", s)
    B = _device(_normal(seed, 1, n, case["nrhs"], nb))
    return dict(case=case, solver=s, B=B, X=torch.zeros_like(B))


def _prepare_uneven(case, seed):
    mats = _members(case, seed)
    batch = UnevenBatch([M.lower_csr(A) for _, A in mats], "SPD", "L",
                        perms=[sds.grid_nd_perm(q, q, 1) for q, _ in mats])
    batch.setparam("amalgamation", (128, 0.25, 8))
    batch.setparam("factor_precision", case["fp"])
    batch.setparam("ir_n_steps", case["ir"])
    batch.execute("analysis")
    batch.execute("factorization")
    graph_capture(batch.solver, nrhs=1)
    B = _device(_normal(seed, 1, batch.n, 1))
    return dict(case=case, batch=batch, B=B, X=torch.zeros_like(B))


def run(state):
    case = state["case"]
    if case["kind"] == "uneven":
        graph_replay(state["batch"].solver, state["X"], state["B"])
        return state["X"]
    s = state["solver"]
    if case.get("op") == "gradient":
        x = SparseSolve.apply(s, state["values"], state["b"])
        dvalues, db = torch.autograd.grad(x, (state["values"], state["b"]), state["xbar"])
        return [x.detach(), dvalues, db]
    if case.get("op") != "solve":
        sds.execute("refactorization", s)
    if case["kind"] == "kkt":
        inertia = sds.getparam(s, "inertia")
        sds.execute("solve", s, state["X"], state["B"])
        return [state["X"], inertia[0], inertia[1]]
    sds.execute("solve", s, state["X"], state["B"])
    if case["kind"] == "lu":
        sds.setparam(s, "solve_mode", 1)
        sds.execute("solve", s, state["Xt"], state["B"])
        sds.setparam(s, "solve_mode", 0)
        return [state["X"], state["Xt"]]
    return state["X"]


# -- the work of a pass ----------------------------------------------------------------------------------

_work = {}


def _analysis(case):
    """(stored factor entries, factorization flops, nnz of the stored matrix, order) of the pattern"""
    if case["kind"] == "uneven":
        tot = np.zeros(4)
        for q, A in _members(case, 1):
            tot += _symbolic(M.lower_csr(A), "SPD", "L", case, perm=sds.grid_nd_perm(q, q, 1),
                             amalgamation=(128, 0.25, 8))
        return tot
    if case["kind"] == "uniform":
        A = M.variable_laplacian((case["nx"], case["ny"]), seed=1)
        return np.array(_symbolic(M.lower_csr(A), "SPD", "L", case)) * case["members"]
    if case["kind"] == "spd":
        A = M.variable_laplacian(_dims(case), seed=1)
        return np.array(_symbolic(M.lower_csr(A), "SPD", "L", case, ordering="algo4" if case["wide"] else "default"))
    if case["kind"] == "kkt":
        K = M.lower_csr(_kkt(case, 1))
        return np.array(_symbolic(K, "S", "L", case, ordering="algo3", values=M.csr_arrays(K)[2],
                                  pivot_pairs="default"))
    return np.array(_symbolic(_lu(case, 1), "G", "F", case))


def _symbolic(A, structure, view, case, amalgamation=None, **kw):
    rp, cv, nz = M.csr_arrays(A)
    amal = amalgamation or ((512, 0.25, 8) if case.get("wide") else (32, 0.25, 8))
    S = sds.symbolic_analysis(rp, cv, A.shape[0], structure, view, "O", amalgamation=amal, **kw)
    f, w = np.asarray(S.front_nrows, dtype=float), np.asarray(S.front_ncols, dtype=float)
    entries = float((f * w - w * (w - 1) / 2).sum())
    return entries, float(S.flops_true), float(nz.size), float(A.shape[0])


def work(case):
    """Factorization: the matrix read, the factor written, its flops (twice for LU: L and U). Each
    solve reads the factor forward and backward, with refinement the matrix and the factor again."""
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _work:
        _work[key] = _analysis(case)
    entries, flops, nnz, n = _work[key]
    es = 8.0 if case["fp"] == "Float64" else 4.0
    sides = 2.0 if case["kind"] == "lu" else 1.0
    nrhs = case.get("nrhs", 1)
    nbytes = ops = 0.0
    if case.get("op") != "solve":
        nbytes += 8.0 * nnz + es * entries * sides
        ops += flops * sides
    # refined solves stop at a tolerance under FGMRES: what its first iteration takes at least
    refine = 1 if case.get("mode") == "fgmres" else case.get("ir", 0)
    solves = (2.0 if case["kind"] == "lu" else 1.0) + refine
    nbytes += solves * 2.0 * es * entries + refine * 12.0 * nnz + 16.0 * n * nrhs
    ops += solves * 4.0 * entries * nrhs
    if case.get("op") == "gradient":
        nbytes += 8.0 * nnz
        ops += nnz
    return {"bytes": float(nbytes), "flops": float(ops)}


# -- 64-bit solutions --------------------------------------------------------------------------------------

def _residual(A, X, B):
    """B - A X with 80-bit products and sums"""
    R = B.astype(np.longdouble)
    values = A.data.astype(np.longdouble)
    for r in range(B.shape[1]):  # (no row of these matrices is empty)
        R[:, r] -= np.add.reduceat(values * X[A.indices, r], A.indptr[:-1])
    return R


def _refined(A, B, solve, steps=4):
    X = np.zeros(B.shape, dtype=np.longdouble)
    for _ in range(steps):
        X = X + solve(_residual(A, X, B).astype(np.float64))
    return X.astype(np.float64)


def _dense_solve(A, *systems):
    """A X = B for each (B, False) of `systems`, A^T X = B for each (B, True)"""
    lu, piv = torch.linalg.lu_factor(torch.tensor(A.toarray()))
    out = []
    for B, transposed in systems:
        out.append(_refined(A.T.tocsr() if transposed else A, B,
                            lambda R: torch.linalg.lu_solve(lu, piv, torch.tensor(R), adjoint=transposed).numpy()))
    return out


def _cg_solve(A, B):
    """Jacobi-preconditioned conjugate gradients in Float64 per right-hand side, refined"""
    n = A.shape[0]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    counts = np.diff(A.indptr)
    width = int(counts.max())
    slot = np.arange(A.indices.size) - np.repeat(A.indptr[:-1], counts)
    rows = np.repeat(np.arange(n), counts)
    cols, vals = np.zeros((width, n), dtype=np.int64), np.zeros((width, n))
    cols[slot, rows] = A.indices
    vals[slot, rows] = A.data
    cols, vals = torch.tensor(cols, device=dev), torch.tensor(vals, device=dev)
    dinv = torch.tensor(1.0 / A.diagonal(), device=dev)[:, None]

    def mul(P):
        Q = vals[0][:, None] * P[cols[0]]
        for e in range(1, width):
            Q += vals[e][:, None] * P[cols[e]]
        return Q

    def solve(Rh):
        R = torch.tensor(Rh, device=dev)
        X = torch.zeros_like(R)
        Z = dinv * R
        P = Z.clone()
        rz = (R * Z).sum(0)
        stop = 1e-20 * rz
        tiny = torch.finfo(torch.float64).tiny
        for it in range(20000):
            Q = mul(P)
            a = rz / (P * Q).sum(0).clamp_min(tiny)
            X += a * P
            R -= a * Q
            Z = dinv * R
            new = (R * Z).sum(0)
            if it % 20 == 19 and bool((new <= stop).all()):
                break
            P = Z + (new / rz.clamp_min(tiny)) * P
            rz = new
        return X.cpu().numpy()

    return _refined(A, B, solve)


def exact(case, seed):
    if case["kind"] == "spd":
        A = M.variable_laplacian(_dims(case), seed=seed)
        A.sort_indices()
        return _cg_solve(A, _normal(seed, 1, A.shape[0], case["nrhs"]))
    if case["kind"] == "kkt":
        K = _kkt(case, seed)
        b = _normal(seed, 1, K.shape[0])
        return [_dense_solve(K, (b[:, None], False))[0][:, 0], None, None]
    if case["kind"] == "lu":
        A = _lu(case, seed)
        n = A.shape[0]
        if n > 14000:  # a dense factorization would take too long
            return None
        if case["op"] == "gradient":
            x, lam = _dense_solve(A, (_normal(seed, 1, n)[:, None], False), (_normal(seed, 2, n)[:, None], True))
            x, lam = x[:, 0], lam[:, 0]
            rows = np.repeat(np.arange(n), np.diff(A.indptr))
            return [x, -lam[rows] * x[A.indices], lam]
        B = _normal(seed, 1, n, case["nrhs"])
        return _dense_solve(A, (B, False), (B, True))
    if case["kind"] == "uniform":
        B = _normal(seed, 1, case["nx"] * case["ny"], case["nrhs"], case["members"])
        X = np.empty_like(B)
        for j, A in enumerate(_uniform(case, seed)):
            X[:, :, j] = _dense_solve(A, (np.ascontiguousarray(B[:, :, j]), False))[0]
        return X
    # conjugate gradients on the block-diagonal matrix of the members
    mats = [A for _, A in _members(case, seed)]
    for A in mats:
        A.sort_indices()
    at = np.concatenate([[0], np.cumsum([A.shape[0] for A in mats])])
    nz = np.concatenate([[0], np.cumsum([A.nnz for A in mats])])
    indices = np.concatenate([A.indices + at[j] for j, A in enumerate(mats)])
    indptr = np.concatenate([A.indptr[:-1] + nz[j] for j, A in enumerate(mats)] + [nz[-1:]])
    whole = type(mats[0])((np.concatenate([A.data for A in mats]), indices, indptr), shape=(at[-1], at[-1]))
    return _cg_solve(whole, _normal(seed, 1, int(at[-1]), 1))
