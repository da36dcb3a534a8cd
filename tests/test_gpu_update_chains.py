"""GPU parity of Schur updates with many contributors and with k loops long
enough to be split into parts: chains of 4-column supernodes (up to 72
contributors, row maps, plain and atomic tiles) and one 1300-column
supernode, under every Schur kernel, against the oracle at the parity bar
(1e-10 relative); edges m = 63, 64, 65, 129 of the output tiles with the
clique pair."""
import numpy as np
import pytest

import sympack_amd as sp
from sympack_amd import matrices as M
from oracle import numeric as onum

pytestmark = pytest.mark.gpu


def _cliques(na, nb, ns):
    """Two dense cliques that share ns nodes, those last."""
    n = na + nb + ns
    rng = np.random.default_rng(n)
    full = np.zeros((n, n))
    for idx in (np.r_[0:na, na + nb:n], np.r_[na:n]):
        full[np.ix_(idx, idx)] = 1.0
    r, c = np.nonzero(np.tril(full))
    v = np.where(r == c, 2.0 * n, -rng.uniform(0.1, 1.0, r.size))
    order = np.lexsort((r, c))
    r, c, v = r[order], c[order], v[order]
    return n, np.searchsorted(c, np.arange(n + 1)), r, v


def _check(gen, ldl, kernel, precision="FP64", **opts):
    n, cp, ri, v = gen()
    A = sp.DistSparseMatrix(n, cp, ri, v)
    m = sp.symPACKMatrix2D()
    m.Init(sp.symPACKOptions(decomposition="LDL" if ldl else "LL", schur_kernel=kernel, precision=precision, **opts))
    m.SymbolicFactorization(A)
    m.DistributeMatrix(A)
    print("case n=%d ldl=%s kernel=%d %s" % (n, ldl, kernel, precision), flush=True)
    m.Factorize()
    B = np.random.default_rng(3).uniform(-1, 1, (n, 2))
    m.Solve(B, 2)
    X = m.GetSolution(2).reshape(n, 2)
    if precision != "FP64":
        assert m.stats()["ir_converged"] == 1 and onum.backward_error(A, X, B) <= 1e-12
        return m
    S = onum.Structure.of(m)
    info, F = onum.factor(S, A, ldl)
    assert info == 0
    Xo = onum.solve(S, F, B, ldl)
    assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) < 1e-10
    return m


@pytest.mark.parametrize("ldl", [False, True], ids=["LL", "LDL"])
@pytest.mark.parametrize("kernel", [0, 1, 2, 3])
def test_long_chains(kernel, ldl):
    rp = sp.RelaxationParameters()
    rp.SetMaxSize(4)
    m = _check(lambda: M.diffusion_3d_7pt(24, seed=5), ldl, kernel, ordering="NDBOX", relax=rp, merge_updates=2)
    assert m.GetUpdateSchedule()[0].max() >= 40  # split into parts


@pytest.mark.parametrize("kernel", [1, 2])
def test_long_chains_fp32_ir(kernel):
    rp = sp.RelaxationParameters()
    rp.SetMaxSize(4)
    _check(lambda: M.diffusion_3d_7pt(24, seed=5), False, kernel, precision="FP32_IR", ordering="NDBOX", relax=rp,
           merge_updates=2)


@pytest.mark.parametrize("kernel", [1, 2, 3])
@pytest.mark.parametrize("na,ns,ldl", [(1300, 129, False), (1300, 65, True), (30, 64, False), (200, 63, True),
                                       (1, 1, False)])
def test_clique_pair(na, ns, ldl, kernel):
    n = na + 40 + ns
    _check(lambda: _cliques(na, 40, ns), ldl, kernel, ordering="NATURAL")
