"""Many narrow supernodes on one etree level (one wave each): widths and rows
around the limits of the two kernels (8 or 16 columns, 56 or 48 rows below),
alone and beside wider ones, LL^T, static LDL^T and FP32 + refinement, against
the oracle at the parity bar (1e-10 relative); a failing pivot in one of
them is reported."""
import numpy as np
import pytest

import sympack_amd as sp
from oracle import numeric as onum

pytestmark = pytest.mark.gpu


def _comb(w, m, count=300, extra=(), top=64, seed=0):
    """`count` cliques of w nodes (and one of every width in `extra`), each
    joined to m nodes of a last clique of `top` nodes."""
    rng = np.random.default_rng(seed)
    widths = [w] * count + list(extra)
    n = sum(widths) + top
    cols = []
    start = 0
    for x in widths:
        below = np.sort(rng.choice(top, m, replace=False)) + n - top
        for j in range(x):
            cols.append(np.r_[start + j:start + x, below])
        start += x
    cols += [np.arange(j, n) for j in range(start, n)]
    rows = np.concatenate(cols)
    colptr = np.r_[0, np.cumsum([len(c) for c in cols])]
    c = np.repeat(np.arange(n), np.diff(colptr))
    v = -rng.uniform(0.1, 1.0, rows.size)
    diag = np.zeros(n)
    np.add.at(diag, rows, -v)
    np.add.at(diag, c, -v)
    v[rows == c] = diag[c[rows == c]] + 1.0
    return sp.DistSparseMatrix(n, colptr, rows, v)


def _run(A, ldl, precision):
    m = sp.symPACKMatrix2D()
    rp = sp.RelaxationParameters(0, 0, 0)
    m.Init(sp.symPACKOptions(ordering="NATURAL", decomposition="LDL" if ldl else "LL", precision=precision, relax=rp))
    m.SymbolicFactorization(A)
    m.DistributeMatrix(A)
    return m


@pytest.mark.parametrize("w,m,extra", [(1, 1, ()), (1, 64, ()), (5, 56, ()), (8, 56, (3, 40)), (8, 57, ()), (9, 48, ()),
                                       (15, 30, (9, 100)), (16, 48, ()), (16, 49, (17,)), (3, 20, (12,) * 260)])
@pytest.mark.parametrize("ldl,precision", [(False, "FP64"), (True, "FP64"), (False, "FP32_IR")])
def test_narrow_levels(w, m, extra, ldl, precision):
    A = _comb(w, m, extra=extra, seed=w * 100 + m)
    print("case w=%d m=%d extra=%s ldl=%s %s" % (w, m, extra[:3], ldl, precision), flush=True)
    M = _run(A, ldl, precision)
    M.Factorize()
    B = np.random.default_rng(1).uniform(-1, 1, (A.size, 3))
    M.Solve(B, 3)
    X = M.GetSolution(3).reshape(A.size, 3)
    if precision != "FP64":
        assert M.stats()["ir_converged"] == 1 and onum.backward_error(A, X, B) <= 1e-12
        return
    S = onum.Structure.of(M)
    info, F = onum.factor(S, A, ldl)
    assert info == 0
    Xo = onum.solve(S, F, B, ldl)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) < 1e-10


@pytest.mark.parametrize("w", [8, 16])
def test_failing_pivot(w):
    A = _comb(w, 10)
    col = 7 * w + w - 1  # last column of the eighth supernode
    A.nzval[A.colptr[col]] = -1.0
    M = _run(A, False, "FP64")
    perm, invp = M.GetOrdering()
    with pytest.raises(sp.NotHPDError) as e:
        M.Factorize()
    assert e.value.column == invp[col]
