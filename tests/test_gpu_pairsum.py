"""The exact 3x3 blocks of A from the noise pair sums, on both sides of the
choice of lanes per item (48 entries an item) and with pixels split into
several items, against the oracle."""
import numpy as np
import pytest

import sanepic_amd
from tests.helpers import make_case, oracle_problem, rel

pytestmark = pytest.mark.gpu


# mean entries a pixel: 32, 64, 128, 1536, 12288; the last two have pixels above one item's 4096
@pytest.mark.parametrize("nside,ndet,nseg,ns", [(4, 2, 3, 1024), (4, 1, 3, 4096), (2, 2, 3, 1024),
                                                (1, 3, 3, 2048), (1, 2, 3, 3 * 2 ** 13)])
def test_blocks_against_the_oracle(nside, ndet, nseg, ns):
    print("pair sums, nside", nside, "ns", ns, flush=True)
    cfg, ds = make_case(nside=nside, ndet=ndet, nseg=nseg, ns=ns)
    P = oracle_problem(cfg, ds)
    ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns)
    ctx.load(cfg, ds)
    ctx.pixelize()
    ctx.setup()
    assert rel(ctx.blocks(), P.exact_blocks()) < 1e-10
    ctx.close()
