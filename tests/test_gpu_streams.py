"""Detectors that share a line of sight are filtered as three streams mixed
bin by bin instead of one stream each.  The operator, chi2 and the iterates
must be the oracle's, which filters every detector, and those of the path with
one stream per detector (taken when the pairs are processed in chunks)."""
import numpy as np
import pytest

import oracle
import sanepic_amd
from sanepic_amd import synth
from tests.helpers import oracle_problem, rel

pytestmark = pytest.mark.gpu

A, B, C = (0.0, 0.0), (0.4, -0.2), (-0.3, 0.45)


def _case(offsets, nseg, ns, nside=16, nan=False):
    tmin = nseg * ns / 19.0 / 60.0
    n = len(offsets)
    cfg = synth.Config(nside=nside, ndet=n, nseg=nseg, ns=ns, fknee=0.2, spin_min=tmin / 40, prec_min=tmin / 5,
                       offsets_deg=offsets, det_angles_deg=[17.0 * k + 3.0 * (k % 3) for k in range(n)])
    ds = synth.make_dataset(cfg, workers=1)
    # every detector its own noise level and slope
    ds["ispf"] = np.stack([synth.ispf_spectrum(ns, cfg.fsamp, 50e-6 * (1 + 0.2 * k), 0.1 + 0.05 * k, 1 + 0.1 * k)
                           for k in range(n)])
    if nan:
        ds["psi"] = ds["psi"].copy()
        ds["psi"][5:9] = np.nan          # filled from the sample before
    return cfg, ds


def _ctx(cfg, ds, precision=sanepic_amd.FP64, split=None, hwp=0, omega=0.0):
    ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns, precision=precision, hwp=hwp, omega=omega)
    ctx.load(cfg, ds)
    ctx.pixelize()
    if split is not None:
        ctx.set_fft_split(split)
    ctx.setup()
    return ctx


@pytest.mark.parametrize("offsets,nseg,ns,split,nline", [
    ([A] * 4, 1, 2 ** 13, None, 1),
    ([A] * 5, 3, 2 ** 14, 9, 1),
    ([A] * 16, 2, 2 ** 13, 9, 1),
    ([B] * 6, 5, 2 ** 15, 10, 1),
    ([A] * 4, 3, 2 ** 16, 12, 1),
    ([A] * 4, 2, 2 ** 17, 9, 1),
    ([A, B, A, B, C, B, A, B, A], 3, 2 ** 14, 10, 3),
    ([B] * 7 + [A, C], 4, 2 ** 16, None, 3),
    ([A] * 4 + [B, C], 3, 2 ** 14, None, 6),  # five streams of six: one per detector
    ([A, B, C, A, B, C], 3, 2 ** 14, None, 6),
])
def test_streams_match_oracle(offsets, nseg, ns, split, nline, monkeypatch):
    print("streams", len(offsets), nseg, ns, split, flush=True)
    cfg, ds = _case(offsets, nseg, ns)
    P = oracle_problem(cfg, ds)
    x = np.random.default_rng(2).standard_normal(3 * P.npix)
    want, c_or = P.apply_A(x), P.chi2(x)
    monkeypatch.setenv("SANEPIC_CHUNK_PAIRS", str(10 ** 6))
    one = _ctx(cfg, ds, split=split)
    per_det, y1 = one.run_records()[0], one.apply(x)
    one.close()
    monkeypatch.delenv("SANEPIC_CHUNK_PAIRS")
    for prec, tol in ((sanepic_amd.FP64, 1e-11), (sanepic_amd.MIXED, 2e-6)):
        ctx = _ctx(cfg, ds, prec, split)
        nrec, used = ctx.run_records()
        assert used
        if len(set(offsets)) == 1:
            assert nrec * len(offsets) == per_det * nline
        elif nline == len(offsets):
            assert nrec == per_det
        else:
            assert nrec < per_det
        y = ctx.apply(x)
        e, e_b, e_1 = rel(y, want), rel(ctx.rhs(), P.rhs()), rel(y, y1)
        print(f"  precision {prec}: A x {e:.1e}, b {e_b:.1e}, against one stream per detector {e_1:.1e}", flush=True)
        assert e < tol and e_b < 1e-11 and e_1 < tol
        assert abs(ctx.chi2(x) - c_or) / c_or < 1e-10
        assert np.array_equal(ctx.apply(x), y)
        ctx.close()


@pytest.mark.parametrize("hwp,nan", [(1, False), (0, True), (1, True)])
def test_streams_hwp_and_missing_pointing(hwp, nan):
    """A half-wave plate's angles are rounded per detector: one stream each."""
    omega = 0.0371
    cfg, ds = _case([B] * 4 + [A] * 4, 3, 2 ** 14, nan=nan)
    P = oracle_problem(cfg, ds, hwp=hwp, omega=omega)
    x = np.random.default_rng(3).standard_normal(3 * P.npix)
    ctx = _ctx(cfg, ds, hwp=hwp, omega=omega)
    assert np.array_equal(ctx.all_pixels(), P.pixels()[0])
    e = rel(ctx.apply(x), P.apply_A(x))
    print(f"  hwp {hwp} nan {nan}: A x {e:.1e}", flush=True)
    assert e < 1e-11
    ctx.close()


def test_first_sample_without_pointing_keeps_the_detectors_apart():
    """Sample 0 of detector 0 has no pixel before it (pixel 0); that of detector
    k takes detector k-1's last pixel, so the detectors' pixels differ and each
    keeps its own stream (its angle is NaN, and so are the products)."""
    cfg, ds = _case([A] * 4, 2, 2 ** 13)
    ds["dec"] = ds["dec"].copy()
    ds["dec"][0] = np.nan
    P = oracle_problem(cfg, ds)
    x = np.random.default_rng(4).standard_normal(3 * P.npix)
    ctx = _ctx(cfg, ds)
    assert np.array_equal(ctx.all_pixels(), P.pixels()[0])
    assert ctx.run_records()[0] >= cfg.ndet * cfg.nseg * cfg.ns // 16
    assert np.isnan(P.apply_A(x)).any() and np.isnan(ctx.apply(x)).any()
    ctx.close()


def test_streams_solve_graph_and_recalibration():
    cfg, ds = _case([A] * 5, 3, 2 ** 15)
    P = oracle_problem(cfg, ds)
    ctx = _ctx(cfg, ds)
    runs = []
    for graph in (False, True):
        ctx.solve_begin(sanepic_amd.PRECOND_BLOCK3, 10, None, True, graph=graph)
        crit = [ctx.step()["crit"] for _ in range(23)]
        runs.append((np.array(crit), ctx.map()))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
    S, _ = ctx.solve(stop=0.0, maxiter=8)
    assert rel(S, P.solve(stop=0.0, maxiter=8)["S"]) < 1e-9
    ctx.close()
    # calibration chosen after the pixelisation: one stream per detector again
    ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns)
    ctx.load(cfg, ds)
    ctx.pixelize()
    n1 = ctx.run_records()[0]
    ctx.set_recalib(True)
    assert ctx.run_records()[0] == 5 * n1
    ctx.setup()
    g = np.random.default_rng(5).uniform(0.8, 1.25, (cfg.ndet, cfg.nseg))
    ctx.set_gains(g)
    P.set_gains(g)
    x = np.random.default_rng(6).standard_normal(3 * P.npix)
    assert rel(ctx.apply(x), P.apply_A(x)) < 1e-11 and rel(ctx.rhs(), P.rhs()) < 1e-11
    ctx.close()
