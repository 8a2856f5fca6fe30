"""Pairs-once kick from 2^20 slots on: PM3's stream joins the pair kernel once it
is done (a second launch that takes parts from the same counters), and the
velocity terms are formed after both.  Clumps beside a sparse field, mixed
levels (PM3 outlasts the pairs) and level 2 (the pairs outlast PM3, and at one
block per CU most of them are left to the joining launch): the kick without the
join (PP after PM3) bit for bit, eager, recorded and replayed, plain and with the
learned stand-in."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def large_layout():
    from cube2_amd.geometry import Geometry
    from cube2_amd.layout import build_layout
    g = Geometry(ng=64, nnt=2, nns=2, ratio_cs=4, ngb=8, app=0.05)
    rng = np.random.default_rng(59)
    pos = np.concatenate([rng.uniform(0, 64, (400000, 3)), 21 + rng.normal(0, 1.2, (90000, 3)),
                          45 + rng.normal(0, 0.7, (40000, 3))]) % 64
    lay = build_layout(pos, rng.normal(0, 1, pos.shape).astype(np.float32), g)
    assert lay.n_used >= 1 << 20
    return lay


@pytest.mark.parametrize("levels", [(2, 6, 3, 2, 5, 4), (2,)])
@pytest.mark.parametrize("learned", [False, True])
@pytest.mark.parametrize("mode", ["ref", "fast"])
def test_joined_kick_equals_the_kick_without_it(large_layout, mode, learned, levels):
    import torch
    from cube2_amd import _lib
    from cube2_amd.kick import ShortRangeKick
    from cube2_amd.learned import LearnedPP
    lay = large_layout
    if learned:
        LearnedPP(seed=0).load(40)
    _lib.set_pp_mode({"ref": _lib.PP_REF, "fast": _lib.PP_FAST}[mode])
    k = ShortRangeKick(lay)
    k.set_levels(np.resize(np.array(levels, np.int32), lay.geom.ns3))
    vp0 = k.d_vp.clone()

    def run(graph=False, **tune):
        for key, v in tune.items():
            _lib.set_tuning(_lib.TUNE_NAMES[key], v)
        k.d_vp.copy_(vp0)
        torch.cuda.synchronize()
        _lib.profile(not graph)
        _lib.profile_reset()
        try:
            r = (k.kick_graph if graph else k.kick)(1.3, 0.05, 2e-3, learned=learned)
            stages = _lib.profile_stats()
        finally:
            _lib.profile(False)
            for key in tune:
                _lib.set_tuning(_lib.TUNE_NAMES[key], 0)
        return r, k.vp_host(), stages

    try:
        r0, v0, st = run(kick_overlap=2)
        assert "pp_pairs_help" not in st and "pp_react_zero" in st  # pairs once, alone
        for blocks in (1, 3):
            for graph in (False, True, True):
                r, v, st = run(graph, pp_overlap_blocks=blocks)
                if not graph:
                    assert st["pp_pairs_help"]["launches"] == 1
                    if levels == (2,) and blocks == 1:  # (3 to 5 ms: it had work)
                        assert st["pp_pairs_help"]["ms"] > 0.1
                print(f"{mode} learned {learned} levels {levels} blocks {blocks} graph {graph}: {int((v != v0).sum())} differ, "
                      f"joined {st.get('pp_pairs_help', {}).get('ms', 0.0):.3f} ms", flush=True)
                assert np.array_equal(v.view(np.uint32), v0.view(np.uint32)), (blocks, graph)
                assert r.f2max_pp == r0.f2max_pp and r.f2max_pm3 == r0.f2max_pm3
                assert np.array_equal(r.vmax, r0.vmax)
                assert (r.p_cand, r.p_acc) == (r0.p_cand, r0.p_acc)
                assert np.array_equal(r.ptotal_pp, r0.ptotal_pp)
    finally:
        _lib.set_pp_mode(_lib.PP_REF)
        _lib.lib().cube2_learned_clear()
