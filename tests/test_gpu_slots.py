"""The slot-parallel kernels (halo velocities, drift, slot positions, layout)
where their blocks of consecutive slots meet cells in unusual ways: nearly
empty images (many empty cells between two slots), a cell of several blocks,
slot counts at and around a block, and a ratio_cs whose divisions are not
exact multiplications.  Integer work and copies: bit-exact against the host
layout and the oracle."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "five_particles_64_tiles": dict(ng=128, nnt=4, nns=1, ratio_cs=4, ngb=8, spread=5, clump=0),
    "one_particle": dict(ng=32, nnt=1, nns=1, ratio_cs=4, ngb=8, spread=1, clump=0),
    "cell_of_5000": dict(ng=64, nnt=2, nns=2, ratio_cs=4, ngb=8, spread=300, clump=5000),
    "one_block": dict(ng=32, nnt=1, nns=1, ratio_cs=4, ngb=4, spread=0, clump=1024),
    "past_one_block": dict(ng=32, nnt=1, nns=1, ratio_cs=4, ngb=4, spread=0, clump=1025),
    "ratio_2": dict(ng=32, nnt=2, nns=1, ratio_cs=2, ngb=4, spread=3000, clump=100),
    "ratio_6": dict(ng=72, nnt=2, nns=1, ratio_cs=6, ngb=12, spread=4000, clump=100),
    "halo_wider_than_image": dict(ng=16, nnt=1, nns=1, ratio_cs=4, ngb=24, spread=500, clump=0),
}


@pytest.mark.parametrize("case", list(CASES))
def test_slot_kernels(oracle_lib, case):
    import torch
    from cube2_amd import _lib
    from cube2_amd.drift import drift_device, refresh_halo_velocities, slot_positions_device
    from cube2_amd.geometry import Geometry
    from cube2_amd.layout import build_layout, build_layout_device
    c = dict(CASES[case])
    spread, clump = c.pop("spread"), c.pop("clump")
    g = Geometry(app=0.05, **c)
    rng = np.random.default_rng(21)
    pos = np.concatenate([rng.uniform(0, g.ng, (spread, 3)),
                          9.5 + rng.uniform(0, 0.4, (clump, 3))]) % g.ng
    vel = rng.uniform(-3, 3, pos.shape).astype(np.float32)
    lay = build_layout(pos, vel, g)
    print(f"slots {case}: {pos.shape[0]} particles, {lay.n_used} slots, {lay.rhoc.size} cells", flush=True)
    rhoc, idx, xp, vp, n = build_layout_device(pos, vel, g)
    assert n == lay.n_used
    for got, want in ((rhoc, lay.rhoc), (idx, lay.idx_b_r), (xp, lay.xp), (vp, lay.vp)):
        assert np.array_equal(got.cpu().numpy(), want)
    # positions: the host's decode, wrapped by whole cells
    got = slot_positions_device(rhoc, idx, xp, n, g).cpu().numpy()
    cell = np.floor(lay.decoded_positions() / g.ratio_cs)
    frac = (lay.xp.view(np.uint16).astype(np.float64) + 0.5) / 65536.0
    assert np.array_equal(got, (np.mod(cell, g.nc) + frac) * g.ratio_cs)
    # halo velocities: stale copies take their particle's velocity
    phys = lay.physical_mask()
    stale = torch.from_numpy(np.where(phys[:, None], lay.vp, np.float32(7))).cuda()
    refresh_halo_velocities(rhoc, idx, stale, n, g)
    assert np.array_equal(stale.cpu().numpy(), lay.vp)
    # drift (the oracle needs steps of at most ncb cells)
    dt = float(np.float32(0.9 * g.ratio_cs * min(g.ncb, g.nt) / 3.0 / 2.0))
    vz = float(np.abs(vel[:, 2]).max())
    o = oracle_lib.drift(g, lay.rhoc, lay.idx_b_r, lay.xp, lay.vp, dt, vz)
    r, i, x, v, k = drift_device(rhoc, idx, xp, vp, n, dt, vz, g)
    assert k == o["n"]
    for got, want in ((r, o["rhoc"]), (i, o["idx_b_r"]), (x, o["xp"]), (v, o["vp"])):
        assert np.array_equal(got.cpu().numpy(), want)


def test_rows_that_start_past_gaps():
    """idx_b_r is the slot range's word, not the running count: an image whose
    rows lie with gaps between them gives the same halo copies and positions
    at its own slots."""
    import torch
    from cube2_amd.drift import refresh_halo_velocities, slot_positions_device
    from cube2_amd.geometry import Geometry
    from cube2_amd.layout import build_layout
    g = Geometry(ng=32, nnt=2, nns=1, ratio_cs=4, ngb=4, app=0.05)
    rng = np.random.default_rng(22)
    lay = build_layout(rng.uniform(0, 32, (2500, 3)), rng.normal(0, 1, (2500, 3)).astype(np.float32), g)
    rows = lay.idx_b_r.reshape(-1)
    gap = np.arange(1, rows.size + 1, dtype=np.int64) * 3        # three unused slots before each row
    n = int(rows[-1] + gap[-1])
    starts = np.concatenate([[0], rows[:-1]])
    to = np.concatenate([np.arange(a, b) + d for a, b, d in zip(starts, rows, gap)])
    xp = np.zeros((n, 3), np.int16)
    vp = np.full((n, 3), 5, np.float32)
    phys = lay.physical_mask()
    xp[to], vp[to] = lay.xp, np.where(phys[:, None], lay.vp, np.float32(7))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    rhoc, idx = d(lay.rhoc), d((rows + gap).reshape(lay.idx_b_r.shape))
    xp, vp = d(xp), d(vp)
    refresh_halo_velocities(rhoc, idx, vp, n, g)
    want = np.full((n, 3), 5, np.float32)
    want[to] = lay.vp
    assert np.array_equal(vp.cpu().numpy(), want)
    pos = slot_positions_device(rhoc, idx, xp, n, g).cpu().numpy()[to]
    cell = np.floor(lay.decoded_positions() / g.ratio_cs)
    frac = (lay.xp.view(np.uint16).astype(np.float64) + 0.5) / 65536.0
    assert np.array_equal(pos, (np.mod(cell, g.nc) + frac) * g.ratio_cs)


def test_rows_that_share_their_slots():
    """The halo rows of one periodic tile hold what its physical rows hold, so
    idx_b_r may name the same slots for both: positions and halo velocities of
    an image without the halo rows' copies."""
    import torch
    from cube2_amd.drift import refresh_halo_velocities, slot_positions_device
    from cube2_amd.geometry import Geometry
    from cube2_amd.layout import build_layout
    g = Geometry(ng=32, nnt=1, nns=1, ratio_cs=4, ngb=8, app=0.05)
    rng = np.random.default_rng(23)
    lay = build_layout(rng.uniform(0, 32, (2500, 3)), rng.normal(0, 1, (2500, 3)).astype(np.float32), g)
    rows = lay.rhoc[0].sum(2).astype(np.int64)                   # [k][j]
    src = (np.arange(g.nte) - g.ncb) % g.nt + g.ncb              # a row's physical twin
    phys = np.zeros_like(rows, bool)
    phys[g.ncb:g.ncb + g.nt, g.ncb:g.ncb + g.nt] = True
    end = np.where(phys, rows, 0).reshape(-1).cumsum().reshape(rows.shape)[src][:, src]
    full = lay.idx_b_r[0] - rows                                 # a row's first slot in the whole layout
    of = np.concatenate([np.arange(full[k, j], full[k, j] + rows[k, j])
                         for k, j in np.argwhere(phys)])         # its slots, kept once
    n = of.size
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    rhoc, idx, xp = d(lay.rhoc), d(end[None]), d(lay.xp[of])
    assert n < lay.n_used and int(idx.max()) == n
    own = lay.physical_mask()[of]
    vp = d(np.where(own[:, None], lay.vp[of], np.float32(7)))
    refresh_halo_velocities(rhoc, idx, vp, n, g)
    assert np.array_equal(vp.cpu().numpy(), lay.vp[of])
    pos = slot_positions_device(rhoc, idx, xp, n, g).cpu().numpy()
    cell = np.floor(lay.decoded_positions() / g.ratio_cs)
    frac = (lay.xp.view(np.uint16).astype(np.float64) + 0.5) / 65536.0
    assert np.array_equal(pos, ((np.mod(cell, g.nc) + frac) * g.ratio_cs)[of])
