"""A solve whose work vectors do not fit reports it and leaves the factor
usable: the next solve, with as few right-hand sides as before, allocates its
vectors anew."""
import numpy as np
import pytest
import torch  # before the library, so that both use the HIP runtime torch brings

import sympack_amd as sp
from oracle import numeric as onum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ldl,precision", [(False, "FP64"), (False, "FP32_IR"), (True, "FP32_IR")])
def test_solve_after_a_failed_allocation(ldl, precision):
    n, cp, ri, v = sp.matrices.laplacian_2d_5pt(20)
    A = sp.DistSparseMatrix(n, cp, ri, v)
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="MMD", decomposition="LDL" if ldl else "LL", precision=precision))
    M.SymbolicFactorization(A)
    M.DistributeMatrix(A)
    M.Factorize()
    B = np.random.default_rng(0).uniform(-1, 1, (n, 2))
    print("case ldl=%s %s" % (ldl, precision), flush=True)
    M.Solve(B, 2)
    X = M.GetSolution(2)
    b = torch.zeros(1, dtype=torch.float64, device="cuda")
    with pytest.raises(sp.SymPACKError, match="out of memory"):
        M.SolveDevice(b.data_ptr(), 2 ** 31 - 1)  # vectors of 3.4 and 6.9 TB: refused before anything reads b
    with pytest.raises(ValueError):
        M.GetSolution(1)
    M.Solve(B, 2)
    tol = 1e-14 if precision == "FP64" else 1e-12
    assert onum.backward_error(A, M.GetSolution(2), B) <= tol and onum.backward_error(A, X, B) <= tol
