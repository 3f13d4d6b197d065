"""The halo fill of a stage in one launch: BC patches, cut copies and the
positivity test together where every face halo is set once, the separate
launches in order otherwise.  Against the oracle: the failing cell it reports
(interior, wall, cut and corner cells, and a halo the wall extrapolation alone
makes negative) and the state after a stage."""
import ctypes

import numpy as np
import pytest

from cosa_amd import _lib
from cosa_amd import case as cases
from cosa_amd.case import Case
from parity_util import make_pair, parity

pytestmark = pytest.mark.gpu

NI, NJ, NK = 9, 9, 5


def _case(open_face=False, wall=14, nk=NK, **cfg):
    c = cases.two_block_case(ni=NI, nj=NJ, nk=nk, nlevel=1, distort=0.2, wall=wall, name="halo", **cfg)
    if open_face:   # block 2's last k face is set by nothing
        c.blocks[1].patches.pop()
        c = Case(c.config, c.blocks, c.cuts, c.xyz, name="halo_open")
    return c


def _at(L, b, v, i, j, k):
    n3 = [int(x) for x in L.points(3)]
    im, jm = int(L.imax[b]), int(L.jmax[b])
    return 5 * sum(n3[:b]) + v * n3[b] + (i + 1) + (im + 3) * ((j + 1) + (jm + 3) * (k + 1))


@pytest.mark.parametrize("open_face", [False, True])
@pytest.mark.parametrize("b,i,j,k,what", [
    (0, 1, 1, 1, "energy"), (0, NI - 1, 4, 2, "energy"), (1, 1, NJ - 1, NK - 1, "energy"),
    (1, 5, 4, 1, "density"), (1, 5, 2, 2, "wall"), (0, 3, 2, NK - 1, "wall")])
def test_failing_cell(open_face, b, i, j, k, what):
    c = _case(open_face)
    q0 = c.freestream()
    L = c.levels[0]
    if what == "energy":
        q0[_at(L, b, 4, i, j, k)] = 0.01
    elif what == "density":
        for v in range(4):   # the velocity kept, so that the pressure stays positive
            q0[_at(L, b, v, i, j, k)] *= 1e-12
    else:                    # second cell off the wall: 3 p1 - p2 < 0 in the halo alone
        q0[_at(L, b, 4, i, j, k)] *= 20
    o, oc, g = make_pair(c, q0)
    try:
        where, done = (ctypes.c_int32 * 8)(), (ctypes.c_int32 * 1)()
        rc = o.or_smooth(oc.ptr(), 1, 0, 0, 1, 1, done, where)
        if rc == 0:
            pytest.fail("the planted state passes the oracle's test")
        with pytest.raises(_lib.CosahipError) as e:
            g.smooth(1, False, False, 1, 1)
        assert e.value.code == rc == 5
        assert list(where)[:5] == e.value.info[:5]
        if what == "wall":
            assert e.value.info[3] < 1
    finally:
        g.close()


@pytest.mark.parametrize("open_face", [False, True])
@pytest.mark.parametrize("nk", [2, 3, NK])   # nk 2: one cell thick, launches in order
def test_stages(open_face, nk):
    c = _case(open_face, wall=14 if nk > 2 else 30, nk=nk, irsop=0 if open_face or nk == 2 else 1)
    q0 = c.perturbed(amp=0.02, seed=3)
    o, oc, g = make_pair(c, q0)
    try:
        where, done = (ctypes.c_int32 * 8)(), (ctypes.c_int32 * 1)()
        assert o.or_smooth(oc.ptr(), 1, 0, 0, 2, 1, done, where) == 0
        g.smooth(1, False, False, 2, 1)
        parity(g.download("q", 1), oc[1]["q"], what=f"q nk={nk} open={open_face}")
    finally:
        g.close()


def _read_back_cases():
    irs = {1: dict(irsop=1, cfl=1.0, cfl_irs=1.5), 2: dict(irsop=2, cfl=1.0, cfl_irs=1.5)}
    two = dict(ni=9, nlevel=1, distort=0.2)
    out = [cases.two_block_case(nj=9, nk=2, name=f"thin_symmetry_{m}", **two, **irs[m]) for m in irs]
    out += [cases.two_block_case(nj=2, nk=5, name=f"thin_wall_{m}", **two, **irs[m]) for m in irs]
    out += [cases.naca_case(33, 13, 2, nlevel=1, name=f"naca_2d_{m}", **irs[m]) for m in irs]
    out.append(cases.two_block_case(nj=9, nk=2, wall=1500, name="thin_laminar", viscous=1, reyno=500.0, stemp=0.383,
                                    **two, **irs[1]))
    for m in irs:
        c = cases.two_block_case(nj=9, nk=5, name=f"open_face_{m}", **two, **irs[m])
        c.blocks[1].patches.pop()
        out.append(Case(c.config, c.blocks, c.cuts, c.xyz, name=c.name))
    return out


@pytest.mark.parametrize("c", _read_back_cases(), ids=lambda c: c.name)
def test_stages_that_read_halos(c):
    """Smoothing with the RK update in the last sweep where a stage reads what
    the stage before it left in a halo: symmetry planes and walls of a block
    one cell thick (their second cell is the far halo) and a face that nothing
    sets.  The conservative halos of prim2cons_b, as in the reference."""
    q0 = c.perturbed(amp=0.01, seed=3)
    o, oc, g = make_pair(c, q0)
    try:
        where, done = (ctypes.c_int32 * 8)(), (ctypes.c_int32 * 1)()
        assert o.or_smooth(oc.ptr(), 1, 0, 0, 2, 1, done, where) == 0
        g.smooth(1, False, False, 2, 1)
        parity(g.download("q", 1), oc[1]["q"], what=f"q {c.name}")
    finally:
        g.close()
