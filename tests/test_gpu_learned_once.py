"""The learned kick in a pairs-once pass: the network's cells (fewer than
`occupancy` particles, level 2) are one-sided sources, beside the small cells
of finer subtiles.  With predictions scaled to 1e-20 what is left is the pair
sums: pair counts those of the ordered pass exactly; the network's particles
get none; the others the plain pairs-once kick's force, of the same pairs in
other groups of at most 64 summed in FP32, the groups in FP64: 1e-6 relative
RMS.  occupancy 2 and 65 are left to the ordered pass (the small cells
reach the network's; such cells may be subsorted), 3 and 64 are the range's
ends."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["ref", "fast"])
@pytest.mark.parametrize("levels", [(2,), (2, 6, 2, 3)])
@pytest.mark.parametrize("occupancy", [2, 3, 20, 64, 65])
def test_learned_pairs_once_is_the_ordered_pass(occupancy, levels, mode):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test without a GPU")
    from cube2_amd import _lib
    from cube2_amd.geometry import Geometry
    from cube2_amd.kick import ShortRangeKick
    from cube2_amd.layout import build_layout
    from cube2_amd.learned import LearnedPP
    g = Geometry(ng=64, nnt=2, nns=2, ratio_cs=4, ngb=8, app=0.05)
    rng = np.random.default_rng(17)
    pos = np.concatenate([rng.uniform(0, 64, (30000, 3)), 20 + rng.normal(0, 1.2, (6000, 3)),
                          41 + rng.normal(0, 0.8, (5000, 3))]) % 64
    lay = build_layout(pos, np.zeros(pos.shape, np.float32), g)
    net = LearnedPP(seed=0)
    net.y_scale = 1e-20

    def kick(learned):
        k = ShortRangeKick(lay)
        k.set_levels(np.resize(np.array(levels, np.int32), g.ns3))
        r = k.kick(1.0, 1.0, 1.0, pm3=False, pp=True, learned=learned)
        return k.vp_host()[lay.physical_mask()].astype(np.float64), r

    print(f"learned {mode} occupancy {occupancy} levels {levels}", flush=True)
    net.load(occupancy)
    _lib.set_pp_mode({"ref": _lib.PP_REF, "fast": _lib.PP_FAST}[mode])
    try:
        plain, _ = kick(False)
        once, r1 = kick(True)
        _lib.set_tuning(_lib.TUNE_PP_NEWTON, 2)
        ordered, r2 = kick(True)
    finally:
        _lib.set_tuning(_lib.TUNE_PP_NEWTON, 0)
        _lib.set_pp_mode(_lib.PP_REF)
        _lib.lib().cube2_learned_clear()
    assert (r1.p_cand, r1.p_acc) == (r2.p_cand, r2.p_acc)
    subst = np.abs(ordered).max(1) < 1e-12
    assert subst.any() and not subst.all()
    assert np.abs(once[subst]).max() < 1e-12
    err = np.sqrt(((once - plain)[~subst] ** 2).sum() / (plain[~subst] ** 2).sum())
    print(f"  {subst.sum()} of {subst.size} substituted, P_acc {r1.p_acc}, error {err:.2e}", flush=True)
    assert err < 1e-6
