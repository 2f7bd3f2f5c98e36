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
