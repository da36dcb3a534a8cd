"""Solve sweeps at the edges of their tiles: one supernode of w columns over m
rows (a clique pair), w around the 16-column blocks and the four waves' k
ranges, m around the 16- and 64-row tiles, right-hand sides around the block
of 16; and many narrow supernodes on one level (64-row workgroups).  Against
the oracle at the parity bar (1e-10 relative)."""
import numpy as np
import pytest

import sympack_amd as sp
from sympack_amd import matrices as M
from oracle import numeric as onum
from test_gpu_update_chains import _cliques

pytestmark = pytest.mark.gpu


def _check(gen, nrhs_list, ldl=False, precision="FP64", **opts):
    n, cp, ri, v = gen()
    A = sp.DistSparseMatrix(n, cp, ri, v)
    m = sp.symPACKMatrix2D()
    m.Init(sp.symPACKOptions(decomposition="LDL" if ldl else "LL", precision=precision, **opts))
    m.SymbolicFactorization(A)
    m.DistributeMatrix(A)
    m.Factorize()
    S = onum.Structure.of(m)
    info, F = onum.factor(S, A, ldl)
    assert info == 0
    for nrhs in nrhs_list:
        print("case n=%d ldl=%s %s nrhs=%d" % (n, ldl, precision, nrhs), flush=True)
        B = np.random.default_rng(nrhs).uniform(-1, 1, (n, nrhs))
        m.Solve(B, nrhs)
        X = m.GetSolution(nrhs).reshape(n, nrhs)
        if precision == "FP64":
            Xo = onum.solve(S, F, B, ldl)
            assert np.linalg.norm(X - Xo) / np.linalg.norm(Xo) < 1e-10
        else:
            assert m.stats()["ir_converged"] == 1 and onum.backward_error(A, X, B) <= 1e-12


@pytest.mark.parametrize("w,m", [(1, 1), (15, 17), (16, 47), (17, 48), (33, 63), (64, 1), (95, 65), (97, 31),
                                 (159, 16), (160, 97)])
def test_one_supernode(w, m):
    _check(lambda: _cliques(w, 3, m), [1, 15, 16, 17, 33], ordering="NATURAL")


@pytest.mark.parametrize("ldl", [False, True], ids=["LL", "LDL"])
def test_fp32(ldl):
    _check(lambda: _cliques(97, 30, 50), [1, 17], ldl=ldl, precision="FP32_IR", ordering="NATURAL")


@pytest.mark.parametrize("ldl,precision", [(False, "FP64"), (True, "FP64"), (False, "FP32_IR"), (True, "FP32_IR")])
@pytest.mark.parametrize("w,m", [(161, 1), (320, 64), (321, 33), (479, 130)])
def test_wide_supernode(w, m, ldl, precision):
    """Wider than a panel of 160 columns: partitioned inverse and substitution."""
    _check(lambda: _cliques(w, 30, m), [1, 17, 70], ldl=ldl, precision=precision, ordering="NATURAL")
    if not ldl and precision == "FP64":
        _check(lambda: _cliques(w, 30, m), [1, 17, 70], ordering="NATURAL", solve_inverse=False)


def test_many_narrow_supernodes():
    rp = sp.RelaxationParameters()
    rp.SetMaxSize(150)
    _check(lambda: M.random_laplacian("2d", 97, 3), [1, 19], ordering="NDGRID", relax=rp)
