"""GPU: factors whose launches are wide enough for the rules on tile counts, and
that those rules were taken.

Forty dense blocks of 192 columns, all coupled to a separator of 650 (which the
last block joins in one supernode of 842 columns): 39 update blocks of 650 x 650
into one target, and 39 supernodes of 842 rows whose trailing updates share a
launch.  Of edge 128 an update block has 21 tiles in its lower part, 819 in all,
of edge 64 it has 66; the first trailing launch, of 39 blocks of 778 x 128, has
39 * 25 = 975 tiles of 64.  The factor is compared entry by entry with one formed
block by block in FP64 on the host: in FP32 the 39 subtractions from diagonal
entries of 84 stay within 39 u 84 = 2e-4, 3e-5 of max |L| = 6.6; 1e-4 and, with
u = 1.1e-16, 1e-12 are asked for.  A 128-wide tile left out of one block's
update changes L by 80 times 1e-4 or more, as the oracle shows.
"""
import numpy as np
import pytest
import scipy.linalg as sla

from suitesparse_amd import _lib, cholmod, problems

pytestmark = pytest.mark.gpu

BLOCKS, WIDTH, SEP = 40, 192, 650
TILES_128, TILES_64 = 39 * 21, 39 * 66


def _arrow():
    rng = np.random.default_rng(3)
    s0 = BLOCKS * WIDTH
    n = s0 + SEP
    D = [rng.standard_normal((WIDTH, WIDTH)) / np.sqrt(WIDTH) for _ in range(BLOCKS)]
    D = [np.tril(d, -1) + 4.0 * np.eye(WIDTH) for d in D]
    C = [2.0 * rng.standard_normal((SEP, WIDTH)) / np.sqrt(WIDTH) for _ in range(BLOCKS)]
    S = np.tril(rng.standard_normal((SEP, SEP)) / np.sqrt(SEP), -1) + (4.0 + 2 * BLOCKS) * np.eye(SEP)
    i, x, cnt = [], [], []
    for b in range(BLOCKS):
        for c in range(WIDTH):
            i += [np.arange(b * WIDTH + c, (b + 1) * WIDTH), np.arange(s0, n)]
            x += [D[b][c:, c], C[b][:, c]]
            cnt.append(WIDTH - c + SEP)
    for c in range(SEP):
        i.append(np.arange(s0 + c, n))
        x.append(S[c:, c])
        cnt.append(SEP - c)
    p = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    A = problems.SymMatrix(n=n, p=p, i=np.concatenate(i).astype(np.int64), x=np.concatenate(x))
    return A, D, C, S


def _factor(D, C, S, lost=None):
    """L by supernodes, as CHOLMOD lays them out; lost = (block, row, column): the
    128-wide tile of that block's update is left out."""
    out, U = [], S + np.tril(S, -1).T
    for b in range(BLOCKS):
        Lb = np.linalg.cholesky(D[b] + np.tril(D[b], -1).T)
        Cb = sla.solve_triangular(Lb, C[b].T, lower=True).T
        V = Cb @ Cb.T
        if lost and lost[0] == b:
            V[lost[1]:lost[1] + 128, lost[2]:lost[2] + 128] = 0.0
        U = U - V
        if b < BLOCKS - 1:
            out.append(np.vstack([Lb, Cb]))
    U = np.tril(U)
    root = np.zeros((WIDTH + SEP, WIDTH + SEP))
    root[:WIDTH, :WIDTH], root[WIDTH:, :WIDTH] = Lb, Cb
    root[WIDTH:, WIDTH:] = np.linalg.cholesky(U + np.tril(U, -1).T)
    return np.concatenate([M.T.ravel() for M in out + [root]])


def _analyzed(prec):
    A, D, C, S = _arrow()
    cm = cholmod.Common(nmethods=1, ordering=cholmod.CHOLMOD_NATURAL, precision=prec)
    L = cholmod.analyze(A, cm)
    assert L.nsuper == BLOCKS and np.array_equal(L.Perm, np.arange(A.n))
    L._numeric(cm)
    return A, cm, L, (D, C, S)


def _check_factor(A, cm, L, blocks, tol):
    Lref = _factor(*blocks)
    for rep in range(2):                         # graph capture, then a replay
        assert cholmod.factorize(A, L, cm) and cm.status == cholmod.CHOLMOD_OK
        assert np.abs(L.x - Lref).max() <= tol * np.abs(Lref).max()
    return Lref


def test_a_setting_of_split16_sets_the_tiles(gpu):
    """The 128-wide tiles are chosen for the split-FP16 kernel: without it the
    plan has 64-wide ones, whatever order the options were set in."""
    A, cm, L, blocks = _analyzed("fp32")
    assert L.info()["update_tiles"] == TILES_128
    L.set_split16(False)
    assert L.info()["update_tiles"] == TILES_64
    _check_factor(A, cm, L, blocks, 1e-4)
    L.set_deterministic(True)                    # (a plan of its own, made while split16 is off)
    L.set_deterministic(False)
    L.set_split16(True)
    assert L.info()["update_tiles"] == TILES_128
    _check_factor(A, cm, L, blocks, 1e-4)


def test_a_table_read_back_and_set_leaves_the_plan(gpu):
    """The default table means the default rules, set or not; another table is
    taken as it is."""
    A, cm, L, _ = _analyzed("fp32")
    table = L.tiles()
    L.set_tiles(table)
    assert L.tiles() == table and L.info()["update_tiles"] == TILES_128
    L.set_tiles([64] * len(table))
    assert L.info()["update_tiles"] == TILES_64
    L.set_tiles(table)
    assert L.info()["update_tiles"] == TILES_128


def _launches(L):
    """Update, diagonal, TRSM and trailing launches of the plan."""
    counts, ms = np.zeros(8, dtype=np.int64), np.zeros(4)
    _lib.check("mxc_factor_stats", _lib.lib().mxc_factor_stats(L._num, cholmod._ptr(counts), cholmod._ptr(ms)))
    return counts[:4].tolist()


def test_fp32_update_launch_of_128_wide_tiles(gpu):
    A, cm, L, blocks = _analyzed("fp32")
    assert L.info()["update_tiles"] == TILES_128
    Lref = _check_factor(A, cm, L, blocks, 1e-4)
    for lost in [(0, 0, 0), (5, 256, 128), (38, 512, 0), (20, 384, 384)]:
        assert np.abs(_factor(*blocks, lost) - Lref).max() > 50 * 1e-4 * np.abs(Lref).max()


def test_fp64_tails_in_a_launch_of_975_tiles(gpu):
    """The diagonal blocks of steps 1 and 2 are the tails of the trailing launches
    of 975 and 468 tiles, those of the 842 columns above tails too, except for the
    last one, whose trailing block is below 64 columns: three diagonal launches."""
    A, cm, L, blocks = _analyzed("fp64")
    assert _launches(L)[1] == 3
    _check_factor(A, cm, L, blocks, 1e-12)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_wide_launches(gpu, prec):
    """A 27-point 64^3 system end to end: the residual of a solve, against n u with
    n the largest front, below 10,000 rows (1e-12 and, in FP32 without refinement,
    6e-4)."""
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
