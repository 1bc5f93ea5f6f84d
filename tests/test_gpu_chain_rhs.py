"""GPU: the chained sweeps over every group size of right-hand sides.

A launch takes up to eight columns, in instantiations for 1, 2, 4 and 8, so
1 .. 9, 16 and 17 columns cover every remainder and the split of wider blocks.
Against the per-step sweeps on the same factor: they differ in summation order
only, within 1e-12 (FP64) and 1e-5 (FP32) relative, as n cond u bounds it.  The
dense orders sit at the edges of the 64-column blocks.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from suitesparse_amd import cholmod, problems

pytestmark = pytest.mark.gpu


def _dense(n):
    M = np.random.default_rng(n).standard_normal((n, n))
    T = sp.csc_matrix(np.tril(M @ M.T + n * np.eye(n)))
    return problems.SymMatrix(n=n, p=T.indptr.astype(np.int64), i=T.indices.astype(np.int64), x=T.data)


CASES = {"dense_64": (lambda: _dense(64), cholmod.CHOLMOD_NATURAL),
         "dense_65": (lambda: _dense(65), cholmod.CHOLMOD_NATURAL),
         "dense_333": (lambda: _dense(333), cholmod.CHOLMOD_NATURAL),
         "stencil27_13": (lambda: problems.stencil3d_27pt(13, seed=3), cholmod.CHOLMOD_METIS)}


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("name", CASES)
def test_chain_groups_match_steps(name, prec, gpu):
    make, ordering = CASES[name]
    A = make()
    cm = cholmod.Common(nmethods=1, ordering=ordering, precision=prec)
    L = cholmod.analyze(A, cm)
    assert cholmod.factorize(A, L, cm) and cm.status == cholmod.CHOLMOD_OK
    tol = 1e-12 if prec == "fp64" else 1e-5
    for nrhs in (1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17):
        B = np.random.default_rng(nrhs).uniform(-1, 1, (A.n, nrhs))
        L.set_solve_chain(False)
        X0 = cholmod.solve(cholmod.CHOLMOD_A, L, B, cm)
        L.set_solve_chain(True)
        for rep in range(2):                     # graph capture, then a replay
            X1 = cholmod.solve(cholmod.CHOLMOD_A, L, B, cm)
            for z in range(nrhs):
                d = np.linalg.norm(X1[:, z] - X0[:, z]) / np.linalg.norm(X0[:, z])
                assert d <= tol, (nrhs, z, d)
