"""Contexts cut their device buffers out of slabs of their own: two contexts
side by side do not disturb each other, released blocks are used again, and a
closed context returns its memory."""
import numpy as np
import pytest
import torch

import sanepic_amd
from sanepic_amd import synth
from tests.helpers import make_case

pytestmark = pytest.mark.gpu


def test_contexts_share_nothing_and_return_their_memory():
    cfg, ds = make_case(nside=64, ndet=3, nseg=4, ns=2 ** 16)
    tmin = 2 ** 18 / 19.0 / 60.0
    un = synth.UnevenConfig(64, [2 ** 15, 3 * 2 ** 14, 2 ** 15, 5 * 2 ** 13], 2 ** 18, spin_min=tmin / 40,
                            prec_min=tmin / 5)
    du = synth.make_uneven_dataset(un, workers=1)

    def uniform():
        c = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns)
        c.load(cfg, ds)
        c.pixelize()
        c.setup()
        return c

    def uneven():
        c = sanepic_amd.Context.uneven(un.nside, un.seglen, un.nsamp)
        c.load_uneven(un, du)
        c.pixelize()
        c.setup()
        return c

    free = []
    want = {}
    for k in range(4):
        a, b = uniform(), uneven()
        for name, c in (("uniform", a), ("uneven", b)):
            x = np.random.default_rng(1).standard_normal(3 * c.npix)
            y, chi = c.apply(x), c.chi2(x)
            if name in want:
                assert np.array_equal(y, want[name][0]) and chi == want[name][1]
            want[name] = (y, chi)
        m, _ = a.solve(maxiter=3, stop=0.0)
        b.solve(maxiter=3, stop=0.0)
        x = np.random.default_rng(1).standard_normal(3 * a.npix)
        assert np.array_equal(a.apply(x), want["uniform"][0])
        a.close()
        assert np.array_equal(b.apply(np.random.default_rng(1).standard_normal(3 * b.npix)), want["uneven"][0])
        b.close()
        free.append(torch.cuda.mem_get_info()[0])
    print("  free MiB after each pair:", [f >> 20 for f in free], flush=True)
    assert free[-1] >= free[0] - (64 << 20)
