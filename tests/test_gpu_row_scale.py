"""Equilibration scaling and ||A||_inf (FP32 factor mode) at the edges of the
kernel's blocks of 64 rows, with more entries than a block stages (2048), and
with a zero stored ahead of every diagonal entry (the last one counts), rows and
columns scaled over six decades.

One CG step from an FP32 factor leaves a backward error far above rounding, and
the library reports max |r| / (||A||_inf max |x| + max |b|).  With at most k
entries per row rounding moves that quotient by (k + 2) u, u = 2^-53, on either
side: the library's and the oracle's differ by at most 2 (k + 2) u plus the
quotients' own rounding."""
import numpy as np
import pytest

import sympack_amd as sp
from oracle import numeric as onum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,half,zeros", [(63, 5, False), (64, 5, False), (65, 5, False), (129, 5, False),
                                          (200, 15, False),   # 1984 entries in a block's rows: staged
                                          (200, 16, False),   # 2112: walked in memory
                                          (200, 40, True), (65, 5, True)])
def test_norm_and_scaling(n, half, zeros):
    rng = np.random.default_rng(n + half)
    s = 10.0 ** rng.uniform(-3, 3, n)
    cols = np.concatenate([np.arange(n - k) for k in range(half + 1)])
    rows = np.concatenate([np.arange(n - k) + k for k in range(half + 1)])
    vals = np.where(rows == cols, 2.0 * half + 2.0, -rng.uniform(0.5, 1.0, rows.size)) * s[rows] * s[cols]
    if zeros:
        cols, rows, vals = (np.r_[a, b] for a, b in ((np.arange(n), cols), (np.arange(n), rows), (np.zeros(n), vals)))
    order = np.lexsort((rows, cols))  # stable: the zeros stay ahead of their diagonal entries
    rows, cols, vals = rows[order], cols[order], vals[order]
    A = sp.DistSparseMatrix(n, np.searchsorted(cols, np.arange(n + 1)), rows, vals)
    print("case n=%d half=%d zeros=%s" % (n, half, zeros), flush=True)
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="AMD", precision="FP32_IR", ir_tol=1e-30, ir_max_iter=1))
    M.SymbolicFactorization(A)
    M.DistributeMatrix(A)
    M.Factorize()
    b = rng.standard_normal((n, 3))
    M.Solve(b, 3)
    be = onum.backward_error(A, M.GetSolution(3), b)
    st = M.stats()
    assert st["fp32_shift"] == 0.0  # scaled to a unit diagonal, FP32 Cholesky does not break down
    assert be <= 1e-5  # one step with the right scaling
    k = 2 * half + 1 + zeros
    assert abs(st["backward_error"] - be) <= 2 * (k + 2) * 2.0 ** -53 + 1e-12 * be
