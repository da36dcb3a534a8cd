"""Products with A in the refinement of the FP32 factor: 64 rows a workgroup,
staged up to 2048 entries and walked in memory above, four right-hand sides a
wave and 16 a pass, at the edges of each.

One step from the FP32 factor leaves a residual far above rounding, and the
library reports the largest |r| / (||A||_inf max |x| + max |b|).  Rounding
moves that quotient by at most (k + 2) u on either side, k the most entries of
a row and u = 2^-53: the library's and the oracle's differ by at most
2 (k + 2) u, plus the rounding of the quotients."""
import numpy as np
import pytest

import sympack_amd as sp
from oracle import numeric as onum

pytestmark = pytest.mark.gpu


def _matrix(n, half, extra, arrow):
    """Band of half-width `half`, `extra` pairs beyond it in rows 64..127,
    optionally a full first column; diagonally dominant."""
    pairs = {(i + d, i) for d in range(1, half + 1) for i in range(n - d)}
    pairs |= {(64 + i + half + 5, 64 + i) for i in range(extra)}
    if arrow:
        pairs |= {(i, 0) for i in range(1, n)}
    rc = sorted(((c, r) for r, c in pairs | {(i, i) for i in range(n)}))
    cols, rows = np.array(rc).T
    rng = np.random.default_rng(n + half + extra)
    vals = -rng.uniform(0.5, 1.0, rows.size)
    per_row = np.bincount(rows, minlength=n) + np.bincount(cols, minlength=n) - 1
    vals[rows == cols] = 1.0 * per_row
    return sp.DistSparseMatrix(n, np.searchsorted(cols, np.arange(n + 1)), rows, vals), per_row


@pytest.mark.parametrize("n,half,extra,arrow", [
    (1, 0, 0, False), (63, 3, 0, False), (64, 3, 0, False), (65, 3, 0, False),
    (200, 15, 32, False),   # rows 64..127: 2048 entries, staged
    (200, 15, 33, False),   # 2050: walked in memory
    (2300, 1, 0, True),     # a row longer than the stage
])
@pytest.mark.parametrize("nrhs", [1, 3, 4, 5, 16, 17, 37])
def test_reported_residual(n, half, extra, arrow, nrhs):
    A, per_row = _matrix(n, half, extra, arrow)
    if extra:
        assert per_row[64:128].sum() == 1984 + 2 * extra
    print("case n=%d half=%d extra=%d arrow=%d nrhs=%d" % (n, half, extra, arrow, nrhs), flush=True)
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="AMD", precision="FP32_IR", ir_tol=1e-30, ir_max_iter=1))
    M.SymbolicFactorization(A)
    M.DistributeMatrix(A)
    M.Factorize()
    b = np.random.default_rng(nrhs).standard_normal((n, nrhs))
    M.Solve(b, nrhs)
    x = M.GetSolution(nrhs).reshape(n, nrhs)
    be = onum.backward_error(A, x, b)
    assert be <= 1e-5  # one step
    assert abs(M.stats()["backward_error"] - be) <= 2 * (per_row.max() + 2) * 2.0 ** -53 + 1e-12 * be
