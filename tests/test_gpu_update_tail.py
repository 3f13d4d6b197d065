"""The update that does fixq and the next stage's cons2prim in the same pass
(k-omega, runs without IRS) against the separate passes: the same bits."""
import numpy as np
import pytest

from cosa_amd import case as cases
from cosa_amd.solver import Solve
from parity_util import rans_cases

pytestmark = pytest.mark.gpu


def _cases():
    noirs = cases.two_block_case(ni=17, nj=9, nk=9, nlevel=2, distort=0.2, name="noirs", irsop=0, cfl=1.0)
    hb = cases.two_block_case(ni=9, nj=9, nk=5, nlevel=1, name="hb_noirs", irsop=0, cfl=1.0, nharms=1, harbal=1,
                              omega=0.5)
    return [noirs, hb] + rans_cases()


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("c", _cases(), ids=lambda c: c.name)
def test_same_bits(c, fp32, monkeypatch):
    out = []
    for fused in ("1", "0"):
        monkeypatch.setenv("COSAHIP_FUSED_UPDATE", fused)
        s = Solve(c, device=0, q=c.perturbed(amp=0.002, seed=4))
        try:
            if fp32:
                s.set_precision(1)
            for m in (1, 2):
                s.cycle(m)
            out.append(s.download("q"))
        finally:
            s.close()
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])
