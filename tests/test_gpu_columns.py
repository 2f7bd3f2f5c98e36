"""Column passes of the four-step transform at the edges of their ranges:
radix-3 and radix-5 columns where the choice between side-by-side and
consecutive sub-transforms changes, and per-block gains applied as the model
is gathered, on every kind of column and an odd number of segments."""
import numpy as np
import pytest

import sanepic_amd
from tests.helpers import make_case, oracle_problem, rel

pytestmark = pytest.mark.gpu


def _ctx(cfg, ds, split=None, recal=False, precision=sanepic_amd.FP64):
    ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns, precision=precision)
    ctx.load(cfg, ds)
    ctx.pixelize()
    if split is not None:
        ctx.set_fft_split(split)
    if recal:
        ctx.set_recalib(True)
    ctx.setup()
    return ctx


# columns of M * 128, M * 256 and M * 512 points: the last and first sizes on
# either side of both limits
@pytest.mark.parametrize("ns", [3 * 2 ** 16, 3 * 2 ** 17, 3 * 2 ** 18, 5 * 2 ** 16, 5 * 2 ** 17])
def test_long_radix_columns(ns):
    print("radix columns, ns", ns, flush=True)
    cfg, ds = make_case(nside=16, ndet=1, nseg=3, ns=ns)
    P = oracle_problem(cfg, ds)
    x = np.random.default_rng(13).standard_normal(3 * P.npix)
    ref, c_ref = P.apply_A(x), P.chi2(x)
    for prec, tol in ((sanepic_amd.FP64, 1e-11), (sanepic_amd.MIXED, 2e-6)):
        ctx = _ctx(cfg, ds, 9, precision=prec)
        assert rel(ctx.apply(x), ref) < tol
        assert rel(ctx.rhs(), P.rhs()) < 1e-11
        if prec == sanepic_amd.FP64:
            assert abs(ctx.chi2(x) - c_ref) / c_ref < 1e-10
        ctx.close()


@pytest.mark.parametrize("precision", [sanepic_amd.FP64, sanepic_amd.MIXED])
@pytest.mark.parametrize("ns,split", [(4096, None), (2 ** 14, None), (3 * 2 ** 13, None), (3 * 2 ** 18, 9),
                                      (5 * 2 ** 13, None)])
def test_gains_in_the_gather(ns, split, precision, monkeypatch):
    """The scaled model has the same bits whether the column pass scales it or
    a gather pass of its own does."""
    print("gains, ns", ns, "split", split, "precision", precision, flush=True)
    cfg, ds = make_case(nside=8, ndet=2, nseg=3, ns=ns, dipole=True)
    g = np.random.default_rng(5).uniform(0.8, 1.25, (cfg.ndet, cfg.nseg))
    out = []
    for pregather in ("0", "1"):
        monkeypatch.setenv("SANEPIC_PREGATHER", pregather)
        ctx = _ctx(cfg, ds, split, recal=True, precision=precision)
        ctx.set_gains(g)
        x = np.random.default_rng(6).standard_normal(3 * ctx.npix)
        out.append((ctx.apply(x), ctx.rhs(), ctx.chi2(x)))
        ctx.close()
    P = oracle_problem(cfg, ds)
    P.set_gains(g)
    assert rel(out[0][0], P.apply_A(x)) < (1e-11 if precision == sanepic_amd.FP64 else 2e-6)
    assert all(np.array_equal(u, v) for u, v in zip(*out))
