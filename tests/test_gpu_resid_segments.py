"""Residual tiles cut into k segments whose length follows the level's size,
and the tile pass as the default of viscous runs, against the kernels that
have neither: one pass per direction (COSAHIP_RESIDUAL=split), and the
per-direction arrangements of the viscous fluxes (COSAHIP_VISCOUS).  The
operations per cell are the same, so the residuals are the same bits."""
import numpy as np
import pytest

from cosa_amd import _lib
from cosa_amd import case as cases
from cosa_amd.config import kw_turbulence
from parity_util import TURB

pytestmark = pytest.mark.gpu

# one-plane segments (a small block), short segments with a remainder, and
# blocks large enough for long segments with a remainder and a short block
DIMS = [[(18, 9, 6)], [(98, 86, 50)], [(130, 66, 36)] * 5 + [(34, 10, 4)]]


def _residual(c, q0, monkeypatch, **env):
    from cosa_amd.solver import Solve
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    g = Solve(c, device=0, q=q0)
    for k in env:
        monkeypatch.delenv(k)
    try:
        for f in ("cons2prim", "bc", "cutman_q"):
            g.call(f, 1, _lib.Q)
        g.call("residual", 1)
        return g.download("res")
    finally:
        g.close()


@pytest.mark.parametrize("dims", DIMS, ids=["one_plane", "short", "long"])
def test_segments_same_bits(dims, monkeypatch):
    c = cases.channel_case(dims, nlevel=1, irsop=1, cfl=2.0, cfl_irs=4.0)
    q0 = c.perturbed(amp=0.02, seed=5)
    print(f"{c.ncell()} cells", flush=True)
    ref = _residual(c, q0, monkeypatch, COSAHIP_RESIDUAL="split")
    assert np.array_equal(_residual(c, q0, monkeypatch).view(np.uint64), ref.view(np.uint64))


@pytest.mark.parametrize("eps", [1e-6, 1e-99, 1e-160])
def test_limiter_floor_same_bits(eps, monkeypatch):
    """Uniform lines (zero differences) and limiter constants on both sides of
    the one below which the quotient by the reciprocal would meet subnormals."""
    c = cases.channel_case([(34, 12, 9)], nlevel=1, irsop=1, cfl=2.0, cfl_irs=4.0, epslimf=eps)
    q0 = c.freestream()
    ref = _residual(c, q0, monkeypatch, COSAHIP_RESIDUAL="split")
    got = _residual(c, q0, monkeypatch)
    assert np.isfinite(ref).all()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("mode", ["faces", "march"])
def test_viscous_default_same_bits(mode, monkeypatch):
    c = cases.two_block_case(ni=34, nj=16, nk=13, nlevel=1, distort=0.1, wall=1500, irsop=1, cfl_irs=2.5, cfl=1.5,
                             **kw_turbulence(0.5, 1e5, tu=1e-3, mutfar=0.1, **TURB))
    q0 = c.perturbed(amp=0.02, seed=6)
    ref = _residual(c, q0, monkeypatch, COSAHIP_VISCOUS=mode)
    assert np.array_equal(_residual(c, q0, monkeypatch).view(np.uint64), ref.view(np.uint64))
