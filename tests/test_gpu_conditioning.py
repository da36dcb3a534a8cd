"""Solves with supernodes wider than a panel (160 columns) on ill-conditioned
matrices whose pivots decay inside a panel: one dense supernode, its structure
that of a covariance or a Gram matrix.  FP64 at the parity bar of the suite, a
backward error at most ten times the oracle's (1e-16 at least); on the Gram
matrix a hundred times, since the factor's own TRSM multiplies by inverse
16 x 16 tiles (restated on the host with a solve by plain substitution: 10 to
30 times the oracle's; with inverses of 160 columns over 1e5 times).  FP32 +
refinement converged at 1e-12."""
import numpy as np
import pytest
import torch  # before the library, so that both use the HIP runtime torch brings

import sympack_amd as sp
from oracle import numeric as onum

pytestmark = pytest.mark.gpu


def _dense(K):
    n = len(K)
    cols = [np.arange(j, n) for j in range(n)]
    return sp.DistSparseMatrix(n, np.r_[0, np.cumsum([len(c) for c in cols])], np.concatenate(cols),
                               np.concatenate([K[j:, j] for j in range(n)]))


def _gauss(n, length, shift, seed):
    p = np.sort(np.random.default_rng(seed).uniform(0, 1, n))
    return np.exp(-((p[:, None] - p) / length) ** 2) + shift * np.eye(n)


def _gram(n, seed):
    """Polynomials of degree below 40 at random points, + 1e-8 I."""
    V = np.polynomial.chebyshev.chebvander(np.sort(np.random.default_rng(seed).uniform(-1, 1, n)), 39)
    K = V @ V.T
    return K / np.abs(K).max() + 1e-8 * np.eye(n)


MATRICES = {
    "gauss_1e-6": lambda n, s: _gauss(n, 0.3, 1e-6, s),
    "gauss_1e-10": lambda n, s: _gauss(n, 0.1, 1e-10, s),
    "gram": _gram,
    "gauss_indefinite": lambda n, s: _gauss(n, 0.1, -0.37, s),
}


def _factored(A, ldl, **opts):
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="NATURAL", decomposition="LDL" if ldl else "LL", **opts))
    M.SymbolicFactorization(A)
    assert M.TotalSupernodeCnt() == 1
    M.DistributeMatrix(A)
    M.Factorize()
    return M


@pytest.mark.parametrize("inverse", [True, False], ids=["default", "no_inverse"])
@pytest.mark.parametrize("n", [161, 333, 480])
@pytest.mark.parametrize("name,ldl", [("gauss_1e-6", False), ("gauss_1e-10", False), ("gram", False),
                                      ("gauss_1e-6", True), ("gauss_indefinite", True)])
def test_backward_error(name, ldl, n, inverse):
    K = MATRICES[name](n, n)
    A = _dense(K)
    M = _factored(A, ldl, solve_inverse=inverse)
    bar = 100 if name == "gram" else 10
    S = onum.Structure.of(M)
    info, F = onum.factor(S, A, ldl)
    assert info == 0
    rng = np.random.default_rng(n)
    for nrhs in (1, 17):
        for B in (rng.uniform(-1, 1, (n, nrhs)), K @ rng.uniform(-1, 1, (n, nrhs))):
            M.Solve(B, nrhs)
            X = M.GetSolution(nrhs).reshape(n, nrhs)
            be, be_o = (onum.backward_error(A, x, B) for x in (X, onum.solve(S, F, B, ldl)))
            print("case %s ldl=%s n=%d inverse=%s nrhs=%d: %.2e oracle %.2e" % (name, ldl, n, inverse, nrhs, be, be_o),
                  flush=True)
            assert be <= bar * max(be_o, 1e-16)
    # the allocation-free solve takes the same route
    b = torch.from_numpy(np.ascontiguousarray(B.T)).cuda()
    x = torch.empty_like(b)
    torch.cuda.synchronize()
    M.SolveDeviceNoAlloc(b.data_ptr(), x.data_ptr(), nrhs)
    assert onum.backward_error(A, x.cpu().numpy().T, B) <= bar * max(be_o, 1e-16)


@pytest.mark.parametrize("ldl", [False, True], ids=["LL", "LDL"])
@pytest.mark.parametrize("n,shift,steps", [(333, 1e-3, 30), (480, 1e-5, 9)])
def test_refined(ldl, n, shift, steps):
    """At 480 and 1e-5 a preconditioner by substitution column by column takes 8
    steps, one by inverses of 160 columns 10 (LDL) and 11."""
    K = _gauss(n, 0.3, shift, 1)
    A = _dense(K)
    M = _factored(A, ldl, precision="FP32_IR")
    B = np.random.default_rng(3).uniform(-1, 1, (n, 4))
    M.Solve(B, 4)
    X = M.GetSolution(4).reshape(n, 4)
    st = M.stats()
    print("case refined ldl=%s n=%d shift=%g: %d steps" % (ldl, n, shift, st["ir_iterations"]), flush=True)
    assert st["ir_converged"] == 1 and st["ir_iterations"] <= steps and onum.backward_error(A, X, B) <= 1e-12
