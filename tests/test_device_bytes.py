"""The device-memory estimate of a factor holds the partitioned inverse, a
second arena, only where the solve uses one: not for FP64 static LDL^T, nor
for plans with a supernode wider than 160 columns."""
import numpy as np
import pytest

import sympack_amd as sp


def _bytes(max_size, **opts):
    n, cp, ri, v = sp.matrices.diffusion_3d_7pt(14, seed=1)
    relax = sp.RelaxationParameters()
    relax.SetMaxSize(max_size)
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="NDBOX", relax=relax, **opts))
    M.SymbolicFactorization(sp.DistSparseMatrix(n, cp, ri, v))
    st = M.stats()
    assert (st["max_width"] > 160) == (max_size > 160)
    return M.DeviceBytes(4), st["factor_entries"] * (8 if opts["precision"] == "FP64" else 4)


@pytest.mark.parametrize("max_size,ldl,precision,inverse", [
    (150, False, "FP64", True), (150, True, "FP64", False), (150, False, "FP32_IR", True), (150, True, "FP32_IR", True),
    (400, False, "FP64", False), (400, True, "FP64", False), (400, False, "FP32_IR", False),
    (400, True, "FP32_IR", False)])
def test_second_arena_where_it_is_used(max_size, ldl, precision, inverse):
    opts = dict(decomposition="LDL" if ldl else "LL", precision=precision)
    (with_, arena), (without, _) = (_bytes(max_size, solve_inverse=s, **opts) for s in (True, False))
    if inverse:
        assert arena <= with_ - without <= 1.2 * arena  # and its task list
    else:
        assert with_ == without
