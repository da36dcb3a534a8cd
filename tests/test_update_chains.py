"""The plan's Schur updates along chains, replayed on the dense pattern: with
every supernode's update restricted to its column cut and computed over its
contributors (rows mapped as the plan maps them), every (source supernode,
target entry) pair of the right-looking algorithm occurs exactly once, and
before the target's panel is factored; columns reported as written by one
supernode of the level are written by no other."""
import numpy as np
import pytest

import sympack_amd as sp
from sympack_amd import matrices as M

CASES = [
    ("diff3d_16_w16", lambda: M.diffusion_3d_7pt(16, seed=1), 16, "NDBOX"),
    ("diff3d_20_w48", lambda: M.diffusion_3d_7pt(20, seed=2), 48, "NDBOX"),
    ("st27_13_w20", lambda: M.stencil_3d_27pt(13, seed=3), 20, "NDBOX"),
    ("lap2d_65_w8", lambda: M.random_laplacian("2d", 65, 1), 8, "NDGRID"),
    ("random_spd", lambda: M.random_spd(400, 0.02, 4), 32, "AMD"),
    ("diag", lambda: M.random_spd(7, 0.0, 4), 32, "AMD"),
]


@pytest.mark.parametrize("merge", [0, 1, 2])
@pytest.mark.parametrize("name,gen,maxsize,ordering", CASES, ids=[c[0] for c in CASES])
def test_every_update_once_and_in_time(name, gen, maxsize, ordering, merge):
    n, cp, ri, v = gen()
    rp = sp.RelaxationParameters()
    rp.SetMaxSize(maxsize)
    m = sp.symPACKMatrix2D()
    m.Init(sp.symPACKOptions(ordering=ordering, relax=rp, merge_updates=merge))
    m.SymbolicFactorization(sp.DistSparseMatrix(n, cp, ri, v))
    xs = np.asarray(m.GetSupernodalPartition()) - 1
    xl, lx = m.GetStructure()
    xl, lx = xl - 1, lx - 1
    ns = len(xs) - 1
    w = np.diff(xs)
    lev = m.supernode_levels()
    sup = np.repeat(np.arange(ns), w)
    panel = [lx[xl[I]:xl[I + 1]] for I in range(ns)]
    off = [panel[I][w[I]:] for I in range(ns)]
    nseg, bcut, excl = m.GetUpdateSchedule()
    if merge == 0:
        assert np.all(nseg <= 1) and np.all(bcut == [len(o) for o in off])
    counts = {}  # source supernode -> dense count of (r1, r2) pairs
    writers = {}  # (level, panel) -> supernodes that write it
    for H in range(ns):
        assert (nseg[H] == 0) == (len(off[H]) == 0)
        assert excl[H] <= bcut[H] <= len(off[H])
        for J in np.unique(sup[off[H][:bcut[H]]]):
            assert lev[J] > lev[H], "applied before the target's level"
            writers.setdefault((lev[H], J), []).append(H)
        for s in range(nseg[H]):
            S, rows = m.GetUpdateSegment(H, s, len(off[H]))
            assert (s == 0) == (S == H) and (S == H or lev[S] < lev[H])
            have = rows >= 0
            assert np.array_equal(panel[S][rows[have]], off[H][have])
            assert not np.isin(off[H][~have], panel[S]).any()
            c = counts.setdefault(S, np.zeros((n, n), np.int8) if n <= 1024 else {})
            rr = off[H][have]
            cols = off[H][:bcut[H]][have[:bcut[H]]]
            for r2 in cols:
                r1 = rr[rr >= r2]
                if n <= 1024:
                    c[r1, r2] += 1
                else:
                    for x in r1:
                        c[(x, r2)] = c.get((x, r2), 0) + 1
    for S in range(ns):
        o = off[S]
        if len(o) == 0:
            continue
        c = counts[S]
        if n <= 1024:
            want = np.zeros((n, n), np.int8)
            for i, r2 in enumerate(o):
                want[o[i:], r2] = 1
            assert np.array_equal(c, want), "supernode %d" % S
        else:
            assert len(c) == len(o) * (len(o) + 1) // 2 and set(c.values()) == {1}, "supernode %d" % S
            assert all((o[j], o[i]) in c for i in range(len(o)) for j in range(i, len(o)))
    for H in range(ns):
        for J in np.unique(sup[off[H][:excl[H]]]):
            assert writers[(lev[H], J)] == [H]


def test_long_chains_on_a_large_grid():
    """48^3: the separators' chains are found (up to 8 members) and only their
    last members write beyond them."""
    n, cp, ri, v = M.diffusion_3d_7pt(48, seed=0)
    rp = sp.RelaxationParameters()
    rp.SetMaxSize(150)
    m = sp.symPACKMatrix2D()
    m.Init(sp.symPACKOptions(ordering="NDBOX", relax=rp))
    m.SymbolicFactorization(sp.DistSparseMatrix(n, cp, ri, v))
    nseg, bcut, _ = m.GetUpdateSchedule()
    assert nseg.max() >= 8
