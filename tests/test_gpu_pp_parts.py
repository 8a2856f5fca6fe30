"""The pairs-once pair kernel's work list: a chunk of many candidates in parts,
taken from counters by whatever wavefronts there are.  One block per CU or 64,
beside PM3 (whose stream joins at the end) or after it, in list order or by
cost: the same partial sums in integers, so the same bits.  Chunks of 16
particles are the same pairs in other groups of at most 64 summed in FP32: the
same counts, Delta-v to 1e-6 relative RMS.  From fewer parts than runs of the
list to cells of thousands of particles."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [(2,), (6, 2, 4)])
@pytest.mark.parametrize("n,clump,width", [(3, 0, 1.0), (200, 70, 0.1), (30000, 9000, 0.3), (2000, 20000, 1.5)])
def test_parts_and_joining_streams_give_the_same_sums(n, clump, width, levels):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test without a GPU")
    from cube2_amd import _lib
    from cube2_amd.geometry import Geometry
    from cube2_amd.kick import ShortRangeKick
    from cube2_amd.layout import build_layout
    g = Geometry(ng=64, nnt=2, nns=1, ratio_cs=4, ngb=8, app=0.05)
    rng = np.random.default_rng(29)
    pos = np.concatenate([rng.uniform(0, 64, (n, 3)), 25 + rng.normal(0, width, (clump, 3))]) % 64
    lay = build_layout(pos, np.zeros(pos.shape, np.float32), g)

    def kick(pm3, **tune):
        k = ShortRangeKick(lay)
        k.set_levels(np.resize(np.array(levels, np.int32), g.ns3))
        for key, v in tune.items():
            _lib.set_tuning(_lib.TUNE_NAMES[key], v)
        try:
            r = k.kick(1.0, 1.0, 1.0, pm3=pm3, pp=True)
        finally:
            for key in tune:
                _lib.set_tuning(_lib.TUNE_NAMES[key], 0)
        return k.vp_host()[lay.physical_mask()], (r.p_cand, r.p_acc)

    print(f"parts: {n} + {clump} particles, levels {levels}", flush=True)
    v, cnt = kick(False)
    for tune in (dict(pp_blocks_per_cu=1), dict(pp_blocks_per_cu=64), dict(pp_order=2)):
        v1, c1 = kick(False, **tune)
        assert c1 == cnt and np.array_equal(v1.view(np.uint32), v.view(np.uint32))
    va, ca = kick(True, kick_overlap=2)
    for blocks in (1, 3):
        vb, cb = kick(True, pp_overlap_blocks=blocks)
        assert ca == cb == cnt and np.array_equal(va.view(np.uint32), vb.view(np.uint32))
    vo, co = kick(False, pp_dense_lg=4)
    err = np.sqrt(((vo - v).astype(np.float64) ** 2).sum() / max((v.astype(np.float64) ** 2).sum(), 1e-300))
    print(f"  P_cand {cnt[0]} P_acc {cnt[1]}, chunks of 16 {err:.1e}", flush=True)
    assert co == cnt
    assert err < 1e-6
