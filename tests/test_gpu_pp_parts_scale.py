"""Short parts of the pairs-once pass's chunks (calls of few slots) only where its
fixed point is fine: at a coarse one (a small softening) a particle's sum does
not depend on how many slots there are elsewhere.  The same particles in a call
just below and just above the slot count of short parts: the same bits.  At a
fine one the sums differ by their FP32 groups of at most 64 pairs, 1e-6 relative
RMS."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("app,bits", [(2e-4, 14), (0.05, 30)])
def test_sums_beside_few_and_many_slots(app, bits):
    from cube2_amd.geometry import Geometry
    from cube2_amd.kick import ShortRangeKick
    from cube2_amd.layout import build_layout
    g = Geometry(ng=64, nnt=2, nns=1, ratio_cs=4, ngb=8, app=app)
    rng = np.random.default_rng(53)
    here = rng.uniform(4, 28, (55296, 3))             # in the first tile
    far = rng.uniform(40.5, 55.5, (1 << 20, 3))       # inside the last one, with no halo copies
    n0 = build_layout(here, None, g).n_used
    dv = []
    for slots in ((1 << 20) - 3000, (1 << 20) + 3000):
        pos = np.concatenate([here, far[:slots - n0]])
        lay = build_layout(pos, np.zeros(pos.shape, np.float32), g)
        assert lay.n_used == slots and np.floor(62 - np.log2(10 / app ** 2 * slots)) == bits
        k = ShortRangeKick(lay)
        k.set_levels(np.full(g.ns3, 2, np.int32))
        k.kick(1.0, 1.0, 1.0, pm3=False, pp=True)
        vp, own = k.vp_host(), lay.physical_mask() & (lay.src < here.shape[0])
        out = np.empty((here.shape[0], 3), np.float32)
        out[lay.src[own]] = vp[own]
        dv.append(out)
        print(f"app {app}: {slots} slots, rms {np.sqrt((out.astype(np.float64) ** 2).mean()):.3e}", flush=True)
    if bits < 22:
        assert np.array_equal(dv[0].view(np.uint32), dv[1].view(np.uint32))
    else:
        d = (dv[0].astype(np.float64) - dv[1]) ** 2
        assert np.sqrt(d.sum() / (dv[1].astype(np.float64) ** 2).sum()) < 1e-6
