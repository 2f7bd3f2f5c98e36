"""The row pass of shared lines of sight at every row length: sets alone and
with detectors on their own, in one launch (small contexts, block counts that
three does and does not divide) and in two (above 2^22 pair values, and rows of
4096), odd and even segment counts, against the oracle."""
import numpy as np
import pytest

import sanepic_amd
from tests.helpers import oracle_problem, rel
from tests.test_gpu_streams import A, B, C, _case, _ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offsets,nseg,ns,split,streams", [
    ([A] * 4, 1, 2 ** 13, 9, (3, 1)),
    ([A] * 4 + [B], 1, 2 ** 13, 9, (4, 2)),
    ([A] * 4 + [B], 3, 2 ** 14, 9, (4, 2)),
    ([A] * 4 + [B], 3, 2 ** 14, 10, (4, 2)),
    ([A] * 6 + [B, C], 2, 2 ** 15, 11, (5, 3)),
    ([B] * 5 + [C] * 4 + [A], 5, 2 ** 15, 11, (7, 3)),
    ([A] * 4 + [B], 2, 2 ** 16, 12, (4, 2)),
    ([A] * 4 + [B], 1, 2 ** 18, 10, (4, 2)),
    ([A] * 4 + [B], 17, 2 ** 17, 10, (4, 2)),
])
def test_rows_against_the_oracle(offsets, nseg, ns, split, streams):
    print("rows", len(offsets), nseg, ns, split, flush=True)
    cfg, ds = _case(offsets, nseg, ns)
    P = oracle_problem(cfg, ds, nthreads=8)
    x = np.random.default_rng(12).standard_normal(3 * P.npix)
    want, c_or = P.apply_A(x), P.chi2(x)
    for prec, tol in ((sanepic_amd.FP64, 1e-11), (sanepic_amd.MIXED, 2e-6)):
        ctx = _ctx(cfg, ds, prec, split)
        assert ctx.streams() == streams
        e, e_c = rel(ctx.apply(x), want), abs(ctx.chi2(x) - c_or) / c_or
        print(f"  precision {prec}: A x {e:.1e}, chi2 {e_c:.1e}", flush=True)
        assert e < tol and e_c < 1e-10
        ctx.close()


def _bits(cfg, ds, split, x, recal=False):
    ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns)
    ctx.load(cfg, ds)
    ctx.pixelize()
    if split is not None:
        ctx.set_fft_split(split)
    if recal:
        ctx.set_recalib(True)
    ctx.setup()
    y = ctx.apply(x)
    ctx.close()
    return y


@pytest.mark.parametrize("offsets,nseg,ns,shared,plain", [
    ([A] * 4, 2, 2 ** 13, 9, 9),
    ([A] * 4, 2, 2 ** 16, 10, 12),
    ([A] * 4, 1, 2 ** 18, 10, 12),
    ([A] * 4, 1, 2 ** 19, 12, 12),
    ([A] * 4 + [B], 3, 2 ** 16, 10, 12),
    ([A] * 4 + [B], 17, 2 ** 17, 12, 12),
])
def test_split_of_shared_lines(offsets, nseg, ns, shared, plain):
    """Rows of 1024 where the operator filters sets of streams, unless the
    caller chose; the usual ones when a calibration takes the sharing away."""
    print("split", len(offsets), nseg, ns, flush=True)
    cfg, ds = _case(offsets, nseg, ns, nside=8)
    ctx = _ctx(cfg, ds)
    x = np.random.default_rng(8).standard_normal(3 * ctx.npix)
    ctx.close()
    assert np.array_equal(_bits(cfg, ds, None, x), _bits(cfg, ds, shared, x))
    assert np.array_equal(_bits(cfg, ds, None, x, True), _bits(cfg, ds, plain, x, True))
    if ns == 2 ** 16:
        kept = _bits(cfg, ds, 11, x, True)
        assert not np.array_equal(kept, _bits(cfg, ds, None, x, True))


@pytest.mark.parametrize("nshare,nown,fp64,mixed", [
    (4, 0, (3, 1), (3, 1)),
    (4, 1, (4, 2), (4, 2)),
    (5, 3, (6, 4), (6, 4)),
    (6, 5, (8, 6), (8, 6)),
    (6, 6, (12, 12), (9, 7)),
    (7, 8, (15, 15), (11, 9)),
    (7, 13, (20, 20), (16, 14)),
    (4, 2, (6, 6), (6, 6)),
])
def test_sharing_pays(nshare, nown, fp64, mixed):
    """A detector on its own costs more beside a set: an FP64 context with many
    of them keeps one stream each."""
    off = [A] * nshare + [(0.05 * (k + 1), 0.3 - 0.02 * k) for k in range(nown)]
    cfg, ds = _case(off, 1, 2 ** 13, nside=8)
    for prec, want in ((sanepic_amd.FP64, fp64), (sanepic_amd.MIXED, mixed)):
        ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns, precision=prec)
        ctx.load(cfg, ds)
        ctx.pixelize()
        assert ctx.streams() == want
        ctx.close()
