"""The autotuner's cache tells contexts of equal sizes apart whose operators run
other passes: a shared line of sight, a half-wave plate (one stream each), gains,
a gather pass of its own, pairs in chunks, and entries of earlier kernels."""
import pytest

import sanepic_amd
from tests.test_gpu_streams import A, _case

pytestmark = pytest.mark.gpu


def test_cache_entries_are_not_shared_between_operators(tmp_path, monkeypatch):
    cfg, ds = _case([A] * 4, 2, 2 ** 15)
    cache = str(tmp_path / "tune.txt")

    def tune(env=None, recal=False, **kw):
        for k, v in (env or {}).items():
            monkeypatch.setenv(k, v)
        ctx = sanepic_amd.Context(cfg.nside, cfg.ndet, cfg.nseg, cfg.ns, **kw)
        for k in env or {}:
            monkeypatch.delenv(k)
        ctx.load(cfg, ds)
        npix, _ = ctx.pixelize()
        if recal:
            ctx.set_recalib(True)
        l1, _ = ctx.autotune(cache)
        ctx.close()
        return l1, npix, len(open(cache).read().splitlines())

    # an entry of the format before the passes were told apart
    _, npix, _ = tune()
    arch = open(cache).read().split()[0]
    with open(cache, "w") as f:
        f.write(f"{arch} ns={cfg.ns} ndet=4 nseg=2 npix={npix} precision=0 log2_n1=9 ms=0.0001\n")
    variants = [dict(), dict(hwp=1, omega=0.03), dict(recal=True), dict(env={"SANEPIC_PREGATHER": "1"}),
                dict(env={"SANEPIC_CHUNK_PAIRS": "2"}), dict(env={"SANEPIC_RUNS": "0"})]
    first = []
    for n, v in enumerate(variants):
        l1, np_, lines = tune(**v)
        assert np_ == npix
        first.append((l1, lines))
    print("  lines after each variant:", [n for _, n in first], flush=True)
    assert [n for _, n in first] == [2, 3, 4, 5, 6, 7]  # each measured for itself
    for v, (l1, _) in zip(variants, first):  # and each finds its own again
        assert tune(**v)[::2] == (l1, 7)
