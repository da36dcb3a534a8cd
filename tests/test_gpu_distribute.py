"""DistributeMatrix on the GPU: equilibration scaling and ||A||_inf (FP32
factor mode) at sizes around a multiple of the kernel's blocks of 64 rows, from
host and device values.

One CG step from an FP32 factor leaves a backward error far above rounding;
the library reports max |r| / (||A||_inf max |x| + max |b|).  The residual's
own rounding is at most (entries per row + 2) u (||A||_inf ||x||_inf +
||b||_inf), i.e. 16 u in the quotient with at most 14 entries per row, on
either side: the two quotients differ by at most 32 u plus their own
rounding."""
import numpy as np
import pytest
import torch  # before the library, so that both use the HIP runtime torch brings

import sympack_amd as sp
from oracle import numeric as onum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("device", [False, True], ids=["host", "device"])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1025])
def test_norm_and_scaling(n, device):
    rng = np.random.default_rng(n)
    # band of half-width 5, rows and columns scaled over six decades
    s = 10.0 ** rng.uniform(-3, 3, n)
    cols = np.concatenate([np.arange(n - k) for k in range(min(6, n))])
    rows = np.concatenate([np.arange(n - k) + k for k in range(min(6, n))])
    vals = np.where(rows == cols, 12.0, -rng.uniform(0.5, 1.0, rows.size)) * s[rows] * s[cols]
    order = np.lexsort((rows, cols))
    rows, cols, vals = rows[order], cols[order], vals[order]
    colptr = np.searchsorted(cols, np.arange(n + 1))
    A = sp.DistSparseMatrix(n, colptr, rows, vals)
    print("case n=%d device=%s" % (n, device), flush=True)
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="AMD", precision="FP32_IR", ir_tol=1e-30, ir_max_iter=1))
    M.SymbolicFactorization(A)
    if device:
        v = torch.from_numpy(vals).cuda()
        torch.cuda.synchronize()
        M.DistributeMatrixDevice(v.data_ptr())
    else:
        M.DistributeMatrix(A)
    M.Factorize()
    b = rng.standard_normal((n, 1))
    M.Solve(b, 1)
    x = M.GetSolution(1).reshape(n, 1)
    be = onum.backward_error(A, x, b)
    st = M.stats()
    assert st["fp32_shift"] == 0.0  # scaled to a unit diagonal, FP32 Cholesky does not break down
    assert be <= 1e-5  # one step with the right scaling
    assert abs(st["backward_error"] - be) <= 32 * 2.3e-16 + 1e-12 * be
