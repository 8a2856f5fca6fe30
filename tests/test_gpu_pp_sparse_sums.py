"""Sums of the small PP cells' particles (k_pp_sparse) where the pass's fixed
point is coarse: softenings so small that it holds 2^-12 to 2^-25 of the unit of
force, in a field around a clump (its neighbours' pairs split among wavefronts)
and at the mean density.  The small cells' sums keep what the fixed point cannot
hold, so against a direct sum in FP64 they are no further off than the ordered
pass with its FP32 sums: the pair forces are the same bits, and a sum that adds
less rounding has no larger RMS error (1.05: samples of 1500)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "field": dict(n=20000, clump=15000, levels=(6, 2, 3, 2, 5, 4)),
    "split": dict(n=3000, clump=60000, levels=(6,)),
    "mean": dict(n=64 ** 3 // 2, clump=0, levels=(6, 4, 2, 6, 3)),
}


@pytest.mark.parametrize("app", [4e-3, 1e-4])
@pytest.mark.parametrize("case", list(CASES))
def test_small_cells_sums_are_as_exact_as_fp32(oracle_lib, case, app):
    from cube2_amd import _lib
    from cube2_amd.geometry import APM3, RATIO_SF, Geometry
    from cube2_amd.kick import ShortRangeKick
    from cube2_amd.layout import build_layout
    c = CASES[case]
    g = Geometry(ng=64, nnt=2, nns=2, ratio_cs=4, ngb=8, app=app)
    rng = np.random.default_rng(43)
    pos = np.concatenate([rng.uniform(0, 64, (c["n"], 3)),
                          25.6 + rng.normal(0, 0.9, (c["clump"], 3))]) % 64
    lay = build_layout(pos, np.zeros(pos.shape, np.float32), g)
    k = 62 - np.log2(10 / app ** 2 * lay.n_used)  # the pass's scale, 2^floor(k)
    assert 12 <= np.floor(k) <= 25
    dv = {}
    for name, newton in (("once", 0), ("ordered", 2)):
        kk = ShortRangeKick(lay)
        kk.set_levels(np.resize(np.array(c["levels"], np.int32), g.ns3))
        _lib.set_tuning(_lib.TUNE_NAMES["pp_newton"], newton)
        try:
            r = kk.kick(1.0, 1.0, 1.0, pm3=False, pp=True)
        finally:
            _lib.set_tuning(_lib.TUNE_NAMES["pp_newton"], 0)
        dv[name] = (kk.vp_host().astype(np.float64) * 6 * np.pi, (r.p_cand, r.p_acc))
    assert dv["once"][1] == dv["ordered"][1]
    # the particles of PP cells of at most 2, by strength
    phys = np.flatnonzero(lay.physical_mask())
    at = lay.decoded_positions()[phys]
    tile_of = lambda cell: (cell[:, 2] * g.nnt + cell[:, 1]) * g.nnt + cell[:, 0]  # noqa: E731
    sub3 = np.floor(at / g.ratio_cs).astype(int) // g.ntt
    tile, q = tile_of(sub3 // g.nns), sub3 % g.nns
    lev = kk.ires[((tile * g.nns + q[:, 2]) * g.nns + q[:, 1]) * g.nns + q[:, 0]]
    rcp = np.array([RATIO_SF[kk.ires.reshape(g.ntile, -1)[t] - 1].max() for t in range(g.ntile)])[tile]
    key = np.floor(at / g.ratio_cs * rcp[:, None]).astype(np.int64)
    _, inv, cnt = np.unique((key[:, 2] * 4096 + key[:, 1]) * 4096 + key[:, 0], return_inverse=True,
                            return_counts=True)
    small = np.flatnonzero(cnt[inv] <= 2)
    f = np.abs(dv["ordered"][0][phys]).max(1)
    tested = 0
    for name, part in (("weak", small[f[small] < 3]), ("strong", small[f[small] >= 3])):
        if part.size < 100:
            continue
        sub = rng.choice(part, min(part.size, 1500), replace=False).astype(np.int32)
        truth = oracle_lib.direct_pp_f64(at, g.ng, sub, APM3[lev[sub] - 1].astype(np.float64), app)
        err = {n: np.sqrt(((v[phys][sub] - truth) ** 2).mean()) for n, (v, _) in dv.items()}
        print(f"{case} app {app} k {k:.1f} {name}: {sub.size} particles, error {err}", flush=True)
        assert err["once"] <= 1.05 * err["ordered"], name
        tested += 1
    assert tested
