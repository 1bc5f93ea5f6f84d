"""The work that a program has this library do, as cases that can be timed.

A case names a family of matrices, a size, a precision, a number of right-hand
sides and a mode.  Every family is one of the seeded generators of
suitesparse_amd.problems; every pass goes through suitesparse_amd.cholmod (or
.batch), as a program does that analysed its pattern once and now brings new
values or new right-hand sides:

  factor_solve   factorize (new values) + solve, FP64
  factor_refine  factorize in FP32 + FP64 iterative refinement to the default
                 relative residual of 1e-10
  solve          solve with a factor that the program keeps
  modify         rank-k update of a kept factor, a solve with it, and the
                 downdate that takes it back

b = A x with x drawn first, so x is the solution that every mode is to return.
The ordering and symbolic analysis of a pattern are made once per process and
kept, as a program does whose matrices share a pattern.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from suitesparse_amd import batch, cholmod, problems

ORDERINGS = {"amd": cholmod.CHOLMOD_AMD, "metis": cholmod.CHOLMOD_METIS}


def listed():
    return [
        # the smallest request of the serving mix: latency of one call
        {"name": "grid2d_32_fp64", "family": "grid2d", "side": 32, "ordering": "amd",
         "mode": "factor_solve", "precision": "fp64", "nrhs": 1, "host": False},
        # the plain method, called as a C program calls it: arrays on the host in and out
        {"name": "laplace2d_100_fp64_host", "family": "laplace2d", "side": 100, "ordering": "amd",
         "mode": "factor_solve", "precision": "fp64", "nrhs": 1, "host": True},
        # a 2D request of the serving mix, odd size, several right-hand sides
        {"name": "grid2d_317_ir", "family": "grid2d", "side": 317, "ordering": "amd",
         "mode": "factor_refine", "precision": "fp32", "nrhs": 3, "host": False},
        # a 3D request of the serving mix
        {"name": "grid3d_41_ir", "family": "grid3d", "side": 41, "ordering": "metis",
         "mode": "factor_refine", "precision": "fp32", "nrhs": 5, "host": False},
        # one time step of a variable-coefficient diffusion problem, FP64
        {"name": "diffusion3d_64_fp64", "family": "diffusion3d", "side": 64, "ordering": "metis",
         "mode": "factor_solve", "precision": "fp64", "nrhs": 1, "host": False},
        # the large 3D systems, plain FP64 and the mixed form
        {"name": "stencil27_80_fp64", "family": "stencil27", "side": 80, "ordering": "metis",
         "mode": "factor_solve", "precision": "fp64", "nrhs": 4, "host": False},
        {"name": "stencil27_80_ir", "family": "stencil27", "side": 80, "ordering": "metis",
         "mode": "factor_refine", "precision": "fp32", "nrhs": 4, "host": False},
        # many small systems at once, both precisions
        {"name": "batch_512_fp64", "family": "batch2d", "systems": 512, "ordering": "amd",
         "mode": "factor_solve", "precision": "fp64", "nrhs": 4, "host": False},
        {"name": "batch_512_ir", "family": "batch2d", "systems": 512, "ordering": "amd",
         "mode": "factor_refine", "precision": "fp32", "nrhs": 4, "host": False},
        # many right-hand sides through a kept factor
        {"name": "diffusion3d_64_solve8", "family": "diffusion3d", "side": 64, "ordering": "metis",
         "mode": "solve", "precision": "fp64", "nrhs": 8, "host": False},
        # low-rank change of a kept factor
        {"name": "grid3d_48_modify8", "family": "grid3d", "side": 48, "ordering": "metis",
         "mode": "modify", "precision": "fp64", "nrhs": 1, "host": False, "rank": 8},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    family = rng.choice(["grid2d", "grid2d", "grid3d", "grid3d", "diffusion3d", "stencil27", "batch2d"])
    case = {"family": family, "ordering": "amd" if family in ("grid2d", "batch2d") else "metis"}
    if family == "grid2d":
        case["side"] = _log_int(rng, 32, 512)
    elif family == "batch2d":
        case["systems"] = _log_int(rng, 16, 512)
    elif family == "stencil27":
        case["side"] = rng.randint(12, 72)
    else:
        case["side"] = rng.randint(16, 64)
    modes = ["factor_solve", "factor_solve", "factor_refine", "factor_refine", "solve"]
    if family in ("grid3d", "diffusion3d"):
        modes.append("modify")
    case["mode"] = rng.choice(modes)
    case["precision"] = "fp32" if case["mode"] == "factor_refine" else "fp64"
    case["nrhs"] = 4 if family == "batch2d" else rng.randint(1, 8)
    case["host"] = family == "grid2d" and rng.random() < 0.25
    if case["mode"] == "modify":
        case["nrhs"] = 1
        case["rank"] = rng.randint(1, 8)
    return case


# ---------------------------------------------------------------------------
# matrices, right-hand sides, plans
# ---------------------------------------------------------------------------

def _single(case, seed: int):
    side = case["side"]
    if case["family"] == "laplace2d":
        return problems.laplace2d_5pt(side)
    if case["family"] == "diffusion3d":
        return problems.diffusion3d_7pt(side, seed=seed)
    if case["family"] == "stencil27":
        return problems.stencil3d_27pt(side, seed=seed)
    rng = np.random.default_rng(seed)
    make = problems.grid2d_lognormal if case["family"] == "grid2d" else problems.grid3d_lognormal
    return make(side, rng)


def _systems(case, seed: int):
    # the sizes belong to the case, the values to the seed
    sides, _ = problems.batch_sides(case["systems"])
    rng = np.random.default_rng(seed)
    return [problems.grid2d_lognormal(int(s), rng) for s in sides]


@functools.lru_cache(maxsize=8)
def _perm(family: str, side: int, ordering: str):
    """The fill-reducing ordering of a pattern, made once."""
    A = _single({"family": family, "side": side}, 0)
    cm = cholmod.Common(nmethods=1, ordering=ORDERINGS[ordering])
    L = cholmod.analyze(A, cm)
    perm = L.Perm.copy()
    L.free()
    return perm


def _analyze(case, A, cm):
    cm.nmethods, cm.ordering = 1, cholmod.CHOLMOD_GIVEN
    perm = _perm(case["family"], case["side"], case["ordering"])
    return cholmod.analyze_p(A, perm, cm)


def _matvec(A, X):
    """A X for the symmetric A of which the lower triangle is stored."""
    col = np.repeat(np.arange(A.n), np.diff(A.p))
    off = A.i != col
    Y = np.empty_like(X)
    for r in range(X.shape[1]):
        x = X[:, r]
        Y[:, r] = (np.bincount(A.i, A.x * x[col], A.n)
                   + np.bincount(col[off], A.x[off] * x[A.i[off]], A.n))
    return Y


def _solution(n: int, case, seed: int):
    rng = np.random.default_rng([seed, 1])
    return rng.uniform(-1.0, 1.0, (n, case["nrhs"]))


def _change(case, A, perm, seed: int):
    """C, in the order of the factor: `rank` columns of tril(P A P') times 0.1,
    which lie in the pattern of L."""
    rng = np.random.default_rng([seed, 2])
    ks = np.sort(rng.choice(A.n, size=case["rank"], replace=False))
    pinv = np.empty(A.n, dtype=np.int64)
    pinv[perm] = np.arange(A.n)
    col = np.repeat(np.arange(A.n), np.diff(A.p))
    ps, rows, vals = [0], [], []
    for k in ks:
        j = perm[k]
        down, right = col == j, (A.i == j) & (col != j)
        r = pinv[np.concatenate([A.i[down], col[right]])]
        v = 0.1 * np.concatenate([A.x[down], A.x[right]])
        keep = r >= k
        r, v = r[keep], v[keep]
        o = np.argsort(r)
        rows.append(r[o])
        vals.append(v[o])
        ps.append(ps[-1] + r.size)
    return np.array(ps, dtype=np.int64), np.concatenate(rows), np.concatenate(vals)


def _device(M):
    """Column-major n x k on the GPU."""
    return torch.from_numpy(np.ascontiguousarray(M.T)).cuda().t()


def prepare(case, seed: int):
    cm = cholmod.Common(precision=case["precision"])
    state = {"case": case, "cm": cm}
    if case["family"] == "batch2d":
        mats = _systems(case, seed)
        state["batch"] = batch.analyze_batch(mats, cm)
        A, L = state["batch"].A, state["batch"].L
    else:
        A = _single(case, seed)
        L = _analyze(case, A, cm)
    X = _solution(A.n, case, seed)
    B = _matvec(A, X)
    state.update(A=A, L=L)
    state["values"] = A.x.copy() if case["host"] else torch.from_numpy(A.x.copy()).cuda()
    if case["mode"] in ("solve", "modify"):
        if not cholmod.factorize(A, L, cm, values=state["values"]) or cm.status != cholmod.CHOLMOD_OK:
            raise RuntimeError(f"factorize: status {cm.status}")
    if case["mode"] == "modify":
        p, i, v = state["C"] = _change(case, A, L.Perm, seed)
        for c in range(case["rank"]):
            rows, w = L.Perm[i[p[c]:p[c + 1]]], v[p[c]:p[c + 1]]
            B[rows] += np.outer(w, w @ X[rows])
    state["B"] = np.asfortranarray(B) if case["host"] else _device(B)
    return state


def run(state):
    case, cm, A, L = state["case"], state["cm"], state["A"], state["L"]
    if case["mode"] in ("factor_solve", "factor_refine"):
        if "batch" in state:
            ok = batch.factorize_batch(state["batch"], values=state["values"])
        else:
            ok = cholmod.factorize(A, L, cm, values=state["values"])
        if not ok or cm.status != cholmod.CHOLMOD_OK:
            raise RuntimeError(f"factorize: status {cm.status}")
    if case["mode"] == "factor_refine":
        if "batch" in state:
            X, _ = batch.solve_refine_batch(state["batch"], state["B"])
        else:
            X, _ = cholmod.solve_refine(L, state["B"], cm)
        return {"x": X, "minor": L.minor}
    if case["mode"] == "modify" and not cholmod.updown(True, state["C"], L, cm):
        raise RuntimeError(f"update: status {cm.status}")
    if "batch" in state:
        X = batch.solve_batch(state["batch"], state["B"])
    else:
        X = cholmod.solve(cholmod.CHOLMOD_A, L, state["B"], cm)
    if case["mode"] == "modify" and not cholmod.updown(False, state["C"], L, cm):
        raise RuntimeError(f"downdate: status {cm.status}")
    return {"x": X, "minor": L.minor}


def exact(case, seed: int):
    """The solution b was made from."""
    n = (int(sum(int(s) ** 2 for s in problems.batch_sides(case["systems"])[0])) if case["family"] == "batch2d"
         else case["side"] ** (2 if case["family"] in ("grid2d", "laplace2d") else 3))
    return {"x": _solution(n, case, seed), "minor": None}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _path_work(case, A, L):
    """Flops of one rank-k modification, and the entries of L it changes, for
    the C of seed 0: the columns on the paths from C's columns to the root."""
    p, i, _ = _change(case, A, L.Perm, 0)
    flops, entries, first = 0.0, 0.0, {}
    for c in range(case["rank"]):
        j = int(i[p[c]])
        while True:
            s = int(np.searchsorted(L.super, j, side="right")) - 1
            m = int(L.super[s + 1]) - j
            nsrow, nscol = int(L.pi[s + 1] - L.pi[s]), int(L.super[s + 1] - L.super[s])
            height = np.arange(nsrow - nscol + 1, nsrow - nscol + m + 1)
            flops += float((6 + 4 * height).sum())
            entries += float(height.sum()) - first.get(s, 0.0) if float(height.sum()) > first.get(s, 0.0) else 0.0
            first[s] = max(first.get(s, 0.0), float(height.sum()))
            if nsrow == nscol:
                break
            j = int(L.s[int(L.pi[s]) + nscol])
    return flops, entries


def work(case):
    cm = cholmod.Common()
    if case["family"] == "batch2d":
        b = batch.analyze_batch(_systems(case, 0), cm)
        A, L = b.A, b.L
    else:
        A = _single(case, 0)
        L = _analyze(case, A, cm)
    item = 4 if case["precision"] == "fp32" else 8
    vectors = 2 * 8.0 * A.n * case["nrhs"]
    sweeps = 4.0 * L.lnz * case["nrhs"]
    if case["mode"] == "solve":
        res = {"bytes": item * L.lnz + vectors, "flops": sweeps}
    elif case["mode"] == "modify":
        flops, entries = _path_work(case, A, L)
        res = {"bytes": item * (L.lnz + 4 * entries) + vectors, "flops": 2 * flops + sweeps}
    else:
        # the values in, L and X out; FP32 takes at least one refinement step
        res = {"bytes": 8.0 * A.nnz_lower + item * L.lnz + vectors,
               "flops": L.fl + (2 if case["mode"] == "factor_refine" else 1) * sweeps}
    L.free()
    return res
