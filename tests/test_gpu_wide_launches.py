"""GPU: factors whose launches are wide enough for the rules on tile counts.

The 27-point 64^3 system has a top separator of several thousand columns: its
FP32 update launches hold more than 512 tiles of 128 (and take them), and its FP64 trailing launches hold 512 to 2048 tiles and carry diagonal tails.
Residual norms against n u with n the largest front, below 10,000 rows: 1e-12
(FP64) and 6e-4 (FP32, one solve without refinement); a lost tile shows as 1e-2
or more.
"""
import numpy as np
import pytest

from suitesparse_amd import cholmod, problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_wide_launches(gpu, prec):
    A = problems.stencil3d_27pt(64, seed=5)
    cm = cholmod.Common(nmethods=1, ordering=cholmod.CHOLMOD_METIS, precision=prec)
    L = cholmod.analyze(A, cm)
    col = np.repeat(np.arange(A.n), np.diff(A.p))
    off = A.i != col
    b = np.random.default_rng(1).uniform(-1, 1, A.n)
    for rep in range(2):                         # graph capture, then a replay
        assert cholmod.factorize(A, L, cm) and cm.status == cholmod.CHOLMOD_OK
        x = cholmod.solve(cholmod.CHOLMOD_A, L, b, cm).reshape(-1)
        r = b - np.bincount(A.i, A.x * x[col], A.n) - np.bincount(col[off], A.x[off] * x[A.i[off]], A.n)
        anorm = np.abs(A.x).max() * 27
        err = np.linalg.norm(r) / (anorm * np.linalg.norm(x) + np.linalg.norm(b))
        assert err <= (1e-12 if prec == "fp64" else 6e-4), (rep, err)
