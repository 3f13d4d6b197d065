"""CIRS sweeps with whole lines resident in LDS (k_cirs_il along i,
k_cirs_strip along j and k) against the sweeps that keep the forward pass in
memory (COSAHIP_CIRS_I=iv, COSAHIP_CIRS_JK=plain): tridi's operations in the
same order (src/cosa.f90:2418-2443), so the same bits -- smoothing iterations,
which take the fused RK update and cons2prim, and the sweeps alone on a random
residual.  Blocks with one-cell and odd lines, partial strips, runs of every
remainder, lines long enough for the narrowest strip and lines that do not
fit and take the other kernels."""
import numpy as np
import pytest

from cosa_amd import case as cases
from cosa_amd.config import kw_turbulence
from parity_util import TURB

pytestmark = pytest.mark.gpu

# A channel one cell high is not among them: its walls extrapolate from the far
# halo, which holds conservative values, and the reference's scheme fails the
# positivity test there (9 x 2 x 3 nodes: oracle and GPU at cell (1, -1, 1) of
# the second stage, any irsop); test_one_cell_j_lines has farfields there.
SMALL = [(34, 18, 6), (9, 3, 2), (17, 12, 40), (71, 37, 15)]
LONG = [(4, 330, 3), (3, 5, 420), (1100, 3, 4)]
# j / k lines at the half-CU bound of 8 lines a work-group, its table and padding counted, and the longest for 4
EDGE = [(9, 242, 3), (5, 3, 243), (11, 247, 4), (7, 178, 3), (6, 3, 177), (4, 3, 493)]
TOO_LONG = [(3, 620, 4), (1600, 3, 3)]
IRS = {1: dict(irsop=1, cfl=2.0, cfl_irs=4.0), 2: dict(irsop=2, cfl=2.0, cfl_irs=4.0)}


def _run(c, q0, monkeypatch, **env):
    from cosa_amd.solver import Solve
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    g = Solve(c, device=0, q=q0)
    for k in env:
        monkeypatch.delenv(k)
    try:
        g.smooth(1, False, False, 2, 1)
        q = g.download("q")
        g.upload("res", np.random.default_rng(3).uniform(-1.0, 1.0, g.size("res")))
        g.call("cirs", 1)
        return q, g.download("res")
    finally:
        g.close()


def _compare(c, monkeypatch):
    q0 = c.perturbed(amp=0.005, seed=8)
    print(f"{c.name}: {c.ncell()} cells", flush=True)
    ref = _run(c, q0, monkeypatch, COSAHIP_CIRS_I="iv", COSAHIP_CIRS_JK="plain")
    for a, b in zip(ref, _run(c, q0, monkeypatch)):
        assert np.isfinite(a).all()
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("irsop", [1, 2])
@pytest.mark.parametrize("dims", [SMALL, LONG, EDGE, TOO_LONG], ids=["small", "long", "edge", "too_long"])
def test_euler_same_bits(dims, irsop, monkeypatch):
    _compare(cases.channel_case(dims, nlevel=1, name=f"channels_{irsop}", **IRS[irsop]), monkeypatch)


@pytest.mark.parametrize("irsop", [1, 2])
def test_one_cell_j_lines(irsop, monkeypatch):
    _compare(cases.two_block_case(ni=9, nj=2, nk=4, nlevel=1, distort=0.1, wall=30, name=f"flat_{irsop}",
                                  **IRS[irsop]), monkeypatch)


@pytest.mark.parametrize("irsop", [1, 2])
def test_komega_same_bits(irsop, monkeypatch):
    kw = dict(irsop=irsop, cfl=1.5, cfl_irs=2.5, ratt=1.4, cflt=1.2)
    _compare(cases.two_block_case(ni=34, nj=14, nk=11, nlevel=1, distort=0.1, name=f"komega_{irsop}", wall=1500, **kw,
                                  **kw_turbulence(0.5, 1e5, tu=1e-3, mutfar=0.1, **TURB)), monkeypatch)


@pytest.mark.parametrize("nj", [173, 174, 178, 353])
def test_komega_edge_same_bits(nj, monkeypatch):
    kw = dict(irsop=1, cfl=1.5, cfl_irs=2.5, ratt=1.4, cflt=1.2)
    _compare(cases.two_block_case(ni=6, nj=nj, nk=4, nlevel=1, distort=0.1, name=f"komega_{nj}", wall=1500, **kw,
                                  **kw_turbulence(0.5, 1e5, tu=1e-3, mutfar=0.1, **TURB)), monkeypatch)
