"""The harmonic-balance source of 3 to 11 snapshots: a thread for a cell and
variable of all snapshots up to 9, a thread for a cell and snapshot above."""
import numpy as np
import pytest

from cosa_amd import case as cases
from parity_util import interior_mask, make_pair, parity
from oracle_bind import dp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh", [1, 2, 3, 4, 5])
def test_src_hb(nh):
    c = cases.two_block_case(ni=10, nj=7, nk=4, nlevel=1, harbal=1, nharms=nh, omega=0.7, name=f"src{nh}")
    o, oc, g = make_pair(c, c.perturbed(amp=0.02, seed=nh))
    try:
        r0 = np.random.default_rng(nh).standard_normal(oc[1]["res"].size) * interior_mask(c)
        oc[1]["res"][:] = r0
        g.upload("res", r0)
        o.or_src_hb(oc.ptr(), 1)
        g.call("src_hb", 1)
        m = interior_mask(c)
        parity(g.download("res")[m], oc[1]["res"][m], what=f"src_hb {c.nsnap}")
    finally:
        g.close()
