"""GPU: diagonal blocks of every width class, against dense LAPACK in FP64.

A dense SPD matrix in natural order is one supernode, so its factor is the
dense Cholesky factor: widths at the edges of the 16-column panels, of the
one-wave and one-lane kernels, of the 64-column blocks and of the 384-column
panels.  Tolerances: a backward-stable factorization of a matrix of
condition number below 10 leaves entries within n u of max|L| (u = 1.1e-16
or 6e-8); 1e-13 and 1e-4 bound that for n <= 450.  L L' x = b is then solved
through the inverses of the diagonal blocks, to ten times that.
"""
import numpy as np
import pytest

from suitesparse_amd import cholmod, problems

pytestmark = pytest.mark.gpu

SIZES = [1, 5, 6, 7, 15, 16, 17, 31, 33, 48, 49, 63, 64, 65, 80, 127, 129, 200, 384, 385, 449]


def _dense(n, rng):
    M = rng.standard_normal((n, n)) / np.sqrt(n)
    return M @ M.T + 2.0 * np.eye(n)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", SIZES)
def test_dense_supernode_matches_lapack(gpu, n, precision):
    rng = np.random.default_rng(n)
    A = _dense(n, rng)
    i, j = np.tril_indices(n)
    o = np.lexsort((i, j))
    p = np.concatenate([[0], np.cumsum(np.bincount(j, minlength=n))]).astype(np.int64)
    S = problems.SymMatrix(n=n, p=p, i=i[o].astype(np.int64), x=A[i, j][o])
    cm = cholmod.Common(nmethods=1, ordering=cholmod.CHOLMOD_NATURAL, precision=precision)
    L = cholmod.analyze(S, cm)
    assert L is not None and L.nsuper == 1
    tol = 1e-13 if precision == "fp64" else 1e-4
    Lref = np.linalg.cholesky(A[np.ix_(L.Perm, L.Perm)])
    B = rng.uniform(-1, 1, (n, 3))
    for rep in range(3):                     # graph capture, then replays
        assert cholmod.factorize(S, L, cm) and cm.status == cholmod.CHOLMOD_OK
        Lx = L.x.reshape(n, n).T
        assert np.abs(Lx - Lref).max() <= tol * np.abs(Lref).max()
    X = cholmod.solve(cholmod.CHOLMOD_A, L, B, cm)
    Xref = np.linalg.solve(A, B)
    assert np.linalg.norm(X - Xref) <= 10 * tol * np.linalg.norm(Xref)


@pytest.mark.parametrize("n,bad", [(40, 0), (40, 39), (64, 17), (200, 130), (449, 400)])
def test_dense_supernode_not_posdef(gpu, n, bad):
    rng = np.random.default_rng(n + bad)
    A = _dense(n, rng)
    A[bad, bad] = -1.0
    i, j = np.tril_indices(n)
    o = np.lexsort((i, j))
    p = np.concatenate([[0], np.cumsum(np.bincount(j, minlength=n))]).astype(np.int64)
    S = problems.SymMatrix(n=n, p=p, i=i[o].astype(np.int64), x=A[i, j][o])
    cm = cholmod.Common(nmethods=1, ordering=cholmod.CHOLMOD_NATURAL)
    L = cholmod.analyze(S, cm)
    P = A[np.ix_(L.Perm, L.Perm)]
    k = int(np.nonzero(L.Perm == bad)[0][0])
    assert cholmod.factorize(S, L, cm) and cm.status == cholmod.CHOLMOD_NOT_POSDEF
    assert L.minor == k
    Lx = L.x.reshape(n, n).T
    Lref = np.zeros((n, n))
    if k > 0:
        Lref[:k, :k] = np.linalg.cholesky(P[:k, :k])
        Lref[k:, :k] = np.linalg.solve(Lref[:k, :k], P[k:, :k].T).T
    assert np.abs(Lx - Lref).max() <= 1e-12 * max(np.abs(Lref).max(), 1.0)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,bad", [(4, 2), (12, 4), (40, 0), (64, 17), (200, 130)])
def test_solve_after_not_posdef_is_finite(gpu, n, bad, precision):
    """L is zero from the failing column on; the inverses of the diagonal blocks
    are those of the factorization that went on with a pivot of 1 there, so a
    solve by them is finite: y_t = X_t (b_t - L_t y), x_t = X_t' (y_t - L' x)."""
    rng = np.random.default_rng(n + bad)
    A = _dense(n, rng)
    A[bad, bad] = -1.0
    i, j = np.tril_indices(n)
    o = np.lexsort((i, j))
    p = np.concatenate([[0], np.cumsum(np.bincount(j, minlength=n))]).astype(np.int64)
    S = problems.SymMatrix(n=n, p=p, i=i[o].astype(np.int64), x=A[i, j][o])
    cm = cholmod.Common(nmethods=1, ordering=cholmod.CHOLMOD_NATURAL, precision=precision)
    L = cholmod.analyze(S, cm)
    L._numeric(cm)
    if precision == "fp32":
        L.set_pivot_rho(0.0)
    assert cholmod.factorize(S, L, cm) and cm.status == cholmod.CHOLMOD_NOT_POSDEF
    M = np.tril(A[np.ix_(L.Perm, L.Perm)])
    k = int(np.nonzero(L.Perm == bad)[0][0])
    assert L.minor == k
    for c in range(n):
        M[c, c] = np.sqrt(M[c, c]) if M[c, c] > 0 else 1.0
        M[c + 1:, c] /= M[c, c]
        M[c + 1:, c + 1:] -= np.tril(np.outer(M[c + 1:, c], M[c + 1:, c]))
    blocks = [slice(c, min(c + 64, n)) for c in range(0, n, 64)]
    X = [np.linalg.inv(M[b, b]) for b in blocks]
    M[:, k:] = 0.0
    B = rng.uniform(-1, 1, (n, 2))
    Y = B[L.Perm]
    for t, b in enumerate(blocks):
        Y[b] = X[t] @ (Y[b] - M[b, :b.start] @ Y[:b.start])
    for t, b in reversed(list(enumerate(blocks))):
        Y[b] = X[t].T @ (Y[b] - M[b.stop:, b].T @ Y[b.stop:])
    want = np.empty_like(Y)
    want[L.Perm] = Y
    got = cholmod.solve(cholmod.CHOLMOD_A, L, B, cm)
    tol = 1e-12 if precision == "fp64" else 1e-3
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
