"""The learned kick's pair sums where a pairs-once pass's fixed point is coarse (a
small softening): of the particles that are not the network's they are no
further from a direct sum in FP64 than the ordered pass's FP32 sums.  1.05: a
sample of 2000; at the smaller softening the fixed point, 2^-14 of the unit of
force, would be ten times as far."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("app,bits", [(3e-4, 14), (0.02, 26)])
def test_learned_kick_sums_are_as_exact_as_fp32(oracle_lib, app, bits):
    from cube2_amd import _lib
    from cube2_amd.geometry import APM3, Geometry
    from cube2_amd.kick import ShortRangeKick
    from cube2_amd.layout import build_layout
    from cube2_amd.learned import LearnedPP
    g = Geometry(ng=64, nnt=2, nns=2, ratio_cs=4, ngb=8, app=app)
    rng = np.random.default_rng(47)
    pos = rng.uniform(0, 64, (1 << 19, 3))
    lay = build_layout(pos, np.zeros(pos.shape, np.float32), g)
    assert np.floor(62 - np.log2(10 / app ** 2 * lay.n_used)) == bits
    net = LearnedPP(seed=0)
    net.y_scale = 1e-20
    net.load(32)
    dv = {}
    try:
        for name, newton in (("built in", 0), ("ordered", 2)):
            k = ShortRangeKick(lay)
            k.set_levels(np.resize(np.array((2, 3, 4, 3), np.int32), g.ns3))
            _lib.set_tuning(_lib.TUNE_NAMES["pp_newton"], newton)
            r = k.kick(1.0, 1.0, 1.0, pm3=False, pp=True, learned=True)
            dv[name] = (k.vp_host().astype(np.float64) * 6 * np.pi, (r.p_cand, r.p_acc))
    finally:
        _lib.set_tuning(_lib.TUNE_NAMES["pp_newton"], 0)
        _lib.lib().cube2_learned_clear()
    assert dv["built in"][1] == dv["ordered"][1]
    phys = np.flatnonzero(lay.physical_mask())
    f = np.abs(dv["ordered"][0][phys]).max(1)
    part = np.flatnonzero((f > 1e-12) & (f < 10))
    at = lay.decoded_positions()[phys]
    sub = rng.choice(part, 2000, replace=False).astype(np.int32)
    cell = np.floor(at[sub] / g.ratio_cs).astype(int) // g.ntt
    t, q = cell // g.nns, cell % g.nns
    tile = (t[:, 2] * g.nnt + t[:, 1]) * g.nnt + t[:, 0]
    lev = k.ires[((tile * g.nns + q[:, 2]) * g.nns + q[:, 1]) * g.nns + q[:, 0]]
    truth = oracle_lib.direct_pp_f64(at, g.ng, sub, APM3[lev - 1].astype(np.float64), app)
    err = {n: np.sqrt(((v[phys][sub] - truth) ** 2).mean()) for n, (v, _) in dv.items()}
    print(f"learned app {app} k {bits}: {part.size} particles, error {err}", flush=True)
    assert err["built in"] <= 1.05 * err["ordered"]
