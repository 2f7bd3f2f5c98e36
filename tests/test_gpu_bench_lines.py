"""bench.py reports the operator of shared lines of sight on a line of its own:
its headline filters one stream per detector and counts that operator's bytes."""
import os

import numpy as np
import pytest

import bench
import sanepic_amd
from sanepic_amd import synth

pytestmark = pytest.mark.gpu


def test_headline_and_shared_line(monkeypatch):
    monkeypatch.delenv("SANEPIC_STREAMS", raising=False)
    cfg = synth.Config(nside=16, ndet=4, nseg=3, ns=2 ** 14, fknee=0.2, spin_min=0.5, prec_min=3.0)
    ds = synth.make_dataset(cfg, workers=1)
    pin = sanepic_amd.PinnedInputs(cfg, ds)
    ntot = cfg.ndet * cfg.nseg * cfg.ns
    got = {}
    for shared in (False, True):
        bench.streams_option(shared)
        r = bench.run_solve(cfg, pin, "fp64", "block", False, None, 2, 1, 40, profile=True, keep_map=True)
        got[shared] = bench.operator_figures(r, cfg, ntot, "none", "fp64"), r["map"]
    pin.close()
    assert "SANEPIC_STREAMS" not in os.environ
    (head, m0), (line, m1) = got[False], got[True]
    assert head["streams"] == {"filtered": 4, "lines_of_sight": 4, "detectors": 4}
    assert line["streams"] == {"filtered": 3, "lines_of_sight": 1, "detectors": 4}
    assert head["operator_alg_bytes"] - line["operator_alg_bytes"] == 3 * ntot // 4 * 20
    assert head["run_records"]["records"] == 4 * line["run_records"]["records"]
    # the same 40 iterates but for rounding
    assert np.linalg.norm(m0 - m1) < 1e-6 * np.linalg.norm(m0)
