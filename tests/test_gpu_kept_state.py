"""What a solve keeps between its steps (the gather map that holds the next
direction, the pinned scalars) survives other calls on the context: the iterates
are those of an undisturbed solve, bit for bit.  And the solve over shared lines
of sight, and which contexts share."""
import numpy as np
import pytest

import sanepic_amd
from tests.helpers import oracle_problem, rel
from tests.test_gpu_streams import A, B, _case, _ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nested", ["0", "1"])
@pytest.mark.parametrize("precision", [sanepic_amd.FP64, sanepic_amd.MIXED])
@pytest.mark.parametrize("offsets,ns", [([A] * 5, 2 ** 13), ([A, B], 2 ** 14), ([A, B], 2048)])
def test_calls_between_steps(offsets, ns, precision, nested, monkeypatch):
    print("between steps", len(offsets), ns, precision, nested, flush=True)
    monkeypatch.setenv("SANEPIC_NESTED_MAP", nested)
    cfg, ds = _case(offsets, 3, ns)
    ctx = _ctx(cfg, ds, precision)
    y = np.random.default_rng(21).standard_normal(3 * ctx.npix)
    between = [None, lambda: ctx.apply(y), lambda: ctx.chi2(y), lambda: ctx.true_residual(),
               lambda: (ctx.map(), ctx.rhs())]
    runs = []
    for call in between:
        for graph in (False, True):
            ctx.solve_begin(sanepic_amd.PRECOND_BLOCK3, 4, None, True, graph=graph)
            h = []
            for k in range(13):  # four refresh iterations, replays of both graphs
                h.append(ctx.step())
                if call and k % 3 != 2:
                    call()
            runs.append((np.array([[v[key] for key in ("crit", "crit2", "alpha", "beta")] for v in h]), ctx.map()))
    for h, m in runs[1:]:
        assert np.array_equal(h, runs[0][0]) and np.array_equal(m, runs[0][1])
    ctx.close()


@pytest.mark.parametrize("offsets", [[A] * 6, [B] * 5 + [A]])
def test_mixed_solve_over_shared_lines(offsets):
    """Eight iterations of the mixed solver against the oracle's: FP32 operator,
    FP64 residual in the first."""
    cfg, ds = _case(offsets, 3, 2 ** 14)
    P = oracle_problem(cfg, ds)
    ctx = _ctx(cfg, ds, sanepic_amd.MIXED)
    assert ctx.streams() == ((3, 1) if len(set(offsets)) == 1 else (4, 2))
    S, _ = ctx.solve(stop=0.0, maxiter=8)
    ref = P.solve(stop=0.0, maxiter=8)["S"]
    print(f"  mixed iterates {rel(S, ref):.1e}", flush=True)
    assert rel(S, ref) < 1e-4
    ctx.close()


def test_which_contexts_share():
    def streams(offsets, hwp=0, recal=False, **change):
        cfg, ds = _case(offsets, 2, 2 ** 13)
        for key, (at, v) in change.items():
            ds[key] = ds[key].copy()
            ds[key][at] = v
        ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns, hwp=hwp, omega=0.03 * hwp)
        ctx.load(cfg, ds)
        ctx.pixelize()
        if recal:
            ctx.set_recalib(True)
        n = ctx.streams()
        ctx.close()
        return n

    four = [B] * 4 + [A] * 4
    assert streams(four) == (6, 2)
    assert streams(four, hwp=1) == (8, 8)  # angles rounded per detector
    assert streams(four, recal=True) == (8, 8)
    assert streams(four, psi=(slice(5, 9), np.nan)) == (6, 2)  # filled from the sample before, for all detectors
    assert streams([A] * 4, dec=(0, np.nan)) == (4, 4)  # no pixel before it: the detectors' pixels differ
    assert streams([A] * 4) == (3, 1)
