"""Diagonal solves of the block substitution on both sides of their dispatch:
hundreds of panels on one level, where more than 16 right-hand sides take a
workgroup per 64 of them and fewer one per 16; also beside a supernode wider
than a panel, whose plan corrects its tile solves.  Against the oracle at the
parity bar (1e-10 relative)."""
import numpy as np
import pytest

import sympack_amd as sp
from oracle import numeric as onum
from test_gpu_narrow import _comb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ldl", [False, True], ids=["LL", "LDL"])
@pytest.mark.parametrize("extra", [(), (200,)], ids=["narrow", "wide"])
@pytest.mark.parametrize("w", [5, 24, 40, 90, 150])
def test_many_panels(w, extra, ldl):
    # 140 panels of one width: 280 workgroups of 16 right-hand sides at 17, above
    # the limit of 256
    A = _comb(w, 20, count=140, extra=extra, seed=w)
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="NATURAL", decomposition="LDL" if ldl else "LL",
                             relax=sp.RelaxationParameters(0, 0, 0), solve_inverse=False))
    M.SymbolicFactorization(A)
    M.DistributeMatrix(A)
    M.Factorize()
    S = onum.Structure.of(M)
    info, F = onum.factor(S, A, ldl)
    assert info == 0
    for nrhs in (16, 17, 64, 70):
        print("case w=%d extra=%s ldl=%s nrhs=%d" % (w, extra, ldl, nrhs), flush=True)
        B = np.random.default_rng(nrhs).uniform(-1, 1, (A.size, nrhs))
        M.Solve(B, nrhs)
        Xo = onum.solve(S, F, B, ldl)
        assert np.linalg.norm(M.GetSolution(nrhs) - Xo) / np.linalg.norm(Xo) < 1e-10
