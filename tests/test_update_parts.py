"""A Schur task holds its k part in the bits above the column tile: the parts
of an update are at most as many as those bits count, also for a chain of tens
of thousands of supernodes."""
import numpy as np
import pytest

import sympack_amd as sp

PART_BITS = 31 - 20  # 20 bits of column tile in a non-negative 32-bit field


def _bordered_chains(k, m):
    """Two chains of k nodes, every node joined to the next one and to a border
    of m nodes."""
    n = 2 * k + m
    border = np.arange(2 * k, n)
    cols = [np.r_[i, [i + 1] if (i + 1) % k else [], border] for i in range(2 * k)]
    cols += [np.arange(j, n) for j in border]
    rows = np.concatenate(cols).astype(np.int64)
    return sp.DistSparseMatrix(n, np.r_[0, np.cumsum([len(c) for c in cols])], rows, np.ones(rows.size))


def test_parts_of_a_long_chain():
    k, m = 45000, 10
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="NATURAL", relax=sp.RelaxationParameters(0, 0, 0), merge_updates=2))
    M.SymbolicFactorization(_bordered_chains(k, m))
    nseg, bcut, _ = M.GetUpdateSchedule()
    # each chain's last member carries the whole chain's update of the border
    assert sorted(nseg)[-2] > k - 10
    parts = M.GetUpdateParts()
    assert np.array_equal(parts > 0, nseg > 0)
    assert 1024 < parts.max() <= 1 << PART_BITS


def test_segment_rows_need_room():
    """The library writes one row per off-diagonal row of the supernode: less
    room than that is refused before the call."""
    n, cp, ri, v = sp.matrices.laplacian_2d_5pt(12)
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering="MMD", relax=sp.RelaxationParameters(0, 0, 0)))
    M.SymbolicFactorization(sp.DistSparseMatrix(n, cp, ri, v))
    xs, (xl, _) = M.GetSupernodalPartition(), M.GetStructure()
    m = np.diff(xl) - np.diff(xs)
    I = int(np.argmax(m))
    assert np.array_equal(M.GetUpdateSegment(I, 0, m[I])[1], np.arange(m[I]) + xs[I + 1] - xs[I])
    with pytest.raises(ValueError):
        M.GetUpdateSegment(I, 0, m[I] - 1)
    with pytest.raises(sp.SymPACKError):
        M.GetUpdateSegment(len(m), 0, n)
