"""The prefix sum over cell counts where its form changes: one tile of 2048
counts, one block over several passes of 8192 (up to 32768 counts), three
launches beyond; whole and ragged last passes.  The layout's and the halo
pass's cell starts depend on every count: bit-exact against the host layout."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng,nnt,ngb,ncells", [(32, 1, 8, 1728), (48, 1, 16, 8000), (64, 1, 8, 8000),
                                               (64, 2, 8, 13824), (96, 1, 16, 32768), (112, 1, 8, 32768),
                                               (116, 1, 8, 35937)])
def test_layout_cell_starts(ng, nnt, ngb, ncells):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test without a GPU")
    from cube2_amd.drift import refresh_halo_velocities
    from cube2_amd.geometry import Geometry
    from cube2_amd.layout import build_layout, build_layout_device
    g = Geometry(ng=ng, nnt=nnt, nns=1, ratio_cs=4, ngb=ngb, app=0.05)
    rng = np.random.default_rng(7)
    pos = np.concatenate([rng.uniform(0, ng, (20000, 3)), 5 + rng.normal(0, 0.5, (3000, 3))]) % ng
    vel = rng.uniform(-3, 3, pos.shape).astype(np.float32)
    lay = build_layout(pos, vel, g)
    print(f"scan: {lay.rhoc.size} cells, {lay.n_used} slots", flush=True)
    assert lay.rhoc.size == ncells
    rhoc, idx, xp, vp, n = build_layout_device(pos, vel, g)
    assert n == lay.n_used
    for got, want in ((rhoc, lay.rhoc), (idx, lay.idx_b_r), (xp, lay.xp), (vp, lay.vp)):
        assert np.array_equal(got.cpu().numpy(), want)
    stale = torch.from_numpy(np.where(lay.physical_mask()[:, None], lay.vp, np.float32(7))).cuda()
    refresh_halo_velocities(rhoc, idx, stale, n, g)
    assert np.array_equal(stale.cpu().numpy(), lay.vp)
