"""The pairs-once pass where PP cells hold at most two particles
(k_pp_sparse): images from nearly empty to clumped, subtiles of levels 2 to 6
side by side (stencils of 1 to 6 cells around the same small cells), one tile
and several, ratios of coarse to standard cells other than 4, and a range
whose stencil is too wide for the kernel's packed coordinates (the ordered
pass).  Pair counts are the oracle's exactly (FAST: but for pairs at the very
cutoff).  Delta-v: the pair forces are the oracle's and their sums at least as
accurate, so the error against an FP64 direct sum is at most 1.5 times the
oracle's own (FP32 sums in order: 3e-6 in a clump of 15000) and 1e-6."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "empty_but_five": dict(ng=64, nnt=2, nns=2, ngb=8, n=5, clump=0, levels=(2, 6, 3, 5)),
    "two_in_one_cell": dict(ng=32, nnt=1, nns=1, ngb=8, n=0, clump=2, levels=(6,)),
    "mean_density_level_6_tiles": dict(ng=64, nnt=2, nns=2, ngb=8, n=64 ** 3 // 4, clump=0, levels=(2, 6, 3, 2, 4)),
    "clumps_beside_sparse": dict(ng=64, nnt=2, nns=2, ngb=8, n=20000, clump=15000, levels=(6, 2, 3, 2, 5, 4)),
    "dense_level_2": dict(ng=32, nnt=1, nns=2, ngb=8, n=40000, clump=0, levels=(2, 2, 2, 6)),
    "odd_subtiles": dict(ng=60, nnt=3, nns=1, ngb=4, n=30000, clump=2000, levels=(5, 2, 3)),
    "wide_range": dict(ng=32, nnt=1, nns=1, ngb=8, n=150, clump=0, levels=(2,), scale=250.0),
}


def _rel_rms(a, b):
    return np.sqrt(((a - b) ** 2).sum()) / max(np.sqrt((b ** 2).sum()), 1e-30)


@pytest.mark.parametrize("mode", ["ref", "fast"])
@pytest.mark.parametrize("case", list(CASES))
def test_sparse_cells_match_the_oracle(oracle_lib, case, mode):
    from cube2_amd import _lib
    from cube2_amd.geometry import APM3, RATIO_SF, Geometry, ixyz3
    from cube2_amd.kick import ShortRangeKick
    from cube2_amd.layout import build_layout
    c = dict(CASES[case])
    n, clump, levels, scale = c.pop("n"), c.pop("clump"), c.pop("levels"), c.pop("scale", 1.0)
    g = Geometry(ratio_cs=4, app=0.05, **c)
    rng = np.random.default_rng(41)
    pos = np.concatenate([rng.uniform(0, g.ng, (n, 3)),
                          g.ng * 0.4 + rng.normal(0, 0.05 if clump == 2 else 0.6, (clump, 3))]) % g.ng
    lay = build_layout(pos, np.zeros(pos.shape, np.float32), g)
    k = ShortRangeKick(lay)
    k.set_levels(np.resize(np.array(levels, np.int32), g.ns3))
    apm3 = (APM3 * np.float32(scale)).astype(np.float32)
    print(f"sparse {case} {mode}: {pos.shape[0]} particles, {lay.n_used} slots", flush=True)
    _lib.set_pp_mode({"ref": _lib.PP_REF, "fast": _lib.PP_FAST}[mode])
    try:
        r = k.kick(1.0, 1.0, 1.0, pm3=False, pp=True, apm3=apm3)
    finally:
        _lib.set_pp_mode(_lib.PP_REF)
    o = oracle_lib.pp_force(g, k.ires, ixyz3(g), apm3, RATIO_SF, lay.rhoc, lay.idx_b_r, lay.xp,
                            lay.vp, 1.0, 1.0, 1.0)
    assert r.p_cand == o["p_cand"]
    if mode == "ref":
        assert r.p_acc == o["p_acc"]
    else:
        assert abs(r.p_acc - o["p_acc"]) <= 1e-6 * o["p_acc"] + 2
    got, want = k.vp_host().astype(np.float64), o["vp"].astype(np.float64)
    if scale != 1.0:  # (wider than the halo: no direct sum; 150 particles, short sums)
        assert _rel_rms(got, want) < (1e-6 if mode == "ref" else 1e-3)
        return
    phys = np.flatnonzero(lay.physical_mask())
    sub = rng.choice(phys.size, min(phys.size, 1500), replace=False).astype(np.int32)
    at = lay.decoded_positions()[phys]
    cell = np.floor(at[sub] / g.ratio_cs).astype(int) // g.ntt  # subtile, over the box
    t, q = cell // g.nns, cell % g.nns
    tile = (t[:, 2] * g.nnt + t[:, 1]) * g.nnt + t[:, 0]
    lev = k.ires[((tile * g.nns + q[:, 2]) * g.nns + q[:, 1]) * g.nns + q[:, 0]]
    acc = oracle_lib.direct_pp_f64(at, g.ng, sub, apm3[lev - 1].astype(np.float64), g.app)
    truth = acc / (6 * np.pi)
    e_got, e_oracle = _rel_rms(got[phys][sub], truth), _rel_rms(want[phys][sub], truth)
    print(f"  P_cand {r.p_cand} P_acc {r.p_acc}, Delta-v error {e_got:.2e}, the oracle's {e_oracle:.2e}",
          flush=True)
    assert e_got <= 1.5 * e_oracle + 1e-6
