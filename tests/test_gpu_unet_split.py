"""The network's convolutions split their output channels over blocks on faces
with few tiles; at nside 256 the first levels run all channels in one block and
the deeper ones split.  Checked on one face against the oracle (the faces do
not interact), with the bounds of test_gpu_learn.py: three times the oracle's
own bf16 sensitivity."""
import numpy as np
import pytest

import oracle.unet as ou
import sanepic_amd
from tests.helpers import rel

pytestmark = pytest.mark.gpu


def test_forward_and_gradient_at_nside_256():
    S, f = 256, 7
    rng = np.random.default_rng(0)
    p = np.concatenate([np.concatenate([rng.standard_normal(9 * ci * co) * np.sqrt(2.0 / (9 * ci)),
                                        0.01 * rng.standard_normal(co)]) for ci, co, _ in ou.SPEC])
    p = p.astype(np.float32)
    x = np.zeros((12, S, S, 10), dtype=np.float32)
    dy = np.zeros((12, S, S, 3), dtype=np.float32)
    x[f] = rng.standard_normal((S, S, 10))
    dy[f] = rng.standard_normal((S, S, 3))
    u = sanepic_amd.UNet(S)
    u.set_params(p)
    y, g = u.backward(x, dy)
    x16 = np.zeros((1, S, S, 16))
    x16[..., :10] = x[f]
    yo, go = ou.grads(p.astype(np.float64), x16, dy[f:f + 1].astype(np.float64))
    pp = p * (1 + 1e-7 * rng.standard_normal(p.size))
    yp, gp = ou.grads(pp, x16, dy[f:f + 1].astype(np.float64))
    e, e0 = rel(y[f], yo[0, ..., :3]), rel(yp[0, ..., :3], yo[0, ..., :3])
    eg, eg0 = rel(g, go), rel(gp, go)
    print(f"  forward {e:.2e} (sensitivity {e0:.2e}), gradient {eg:.2e} ({eg0:.2e})", flush=True)
    assert e < 3 * e0 + 1e-4 and e < 3e-2
    assert eg < 3 * eg0 + 1e-3 and eg < 0.3
    u.close()
