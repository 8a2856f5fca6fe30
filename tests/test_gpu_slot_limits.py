"""The slot-parallel kernels at the largest slot counts: every slot is written
where the count ends within a block of 2^31, and images of 2^31 slots and more
have positions and halo velocities.  Copies and decodes: bit-exact."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gives_the_gigabytes_back():
    yield
    import gc

    import torch
    from cube2_amd import _lib
    gc.collect()
    torch.cuda.empty_cache()           # torch's
    _lib.lib().c_gpu_velocity_finalize()  # the library's workspaces


def _geom():
    from cube2_amd.geometry import Geometry
    return Geometry(ng=32, nnt=1, nns=1, ratio_cs=4, ngb=4, app=0.05)


def test_layout_of_nearly_2_31_slots_is_filled_to_its_end():
    """2^28 - 1 particles of the image's corner cell, which the one tile holds
    8 times: 2^31 - 8 slots, 8 runs of the particles in input order."""
    import ctypes as C

    import torch
    from cube2_amd import _lib
    g = _geom()
    n = (1 << 28) - 1
    print(f"layout of {8 * n} slots", flush=True)
    _lib.set_params(g)
    pos = torch.full((n, 3), 0.1, dtype=torch.float64, device="cuda")
    vel = _numbered(n)
    rhoc = torch.empty((1, g.nte, g.nte, g.nte), dtype=torch.int32, device="cuda")
    idx = torch.empty((1, g.nte, g.nte), dtype=torch.int64, device="cuda")
    xp = torch.full((8 * n, 3), -1, dtype=torch.int16, device="cuda")
    vp = torch.full((8 * n, 3), -1.0, dtype=torch.float32, device="cuda")
    used = C.c_int64(0)
    _lib.check(_lib.lib().cube2_layout_build_dev(pos.data_ptr(), vel.data_ptr(), n, rhoc.data_ptr(),
                                                 idx.data_ptr(), xp.data_ptr(), vp.data_ptr(), 8 * n,
                                                 C.byref(used)))
    assert used.value == 8 * n and int(idx[0, -1, -1]) == 8 * n
    code = int(0.1 / g.ratio_cs * 65536)
    for k in range(8):
        assert torch.equal(vp[k * n:(k + 1) * n], vel), k
        assert int(xp[k * n:(k + 1) * n].min()) == code == int(xp[k * n:(k + 1) * n].max()), k


def _corner_image(n):
    """An image whose only particles, n of them, lie in the corner cell, which
    the one tile holds 8 times: (geometry, rhoc, idx_b_r, slots)."""
    import torch
    g = _geom()
    rhoc = torch.zeros((1, g.nte, g.nte, g.nte), dtype=torch.int32, device="cuda")
    at = torch.tensor([g.ncb, g.ncb + g.nt], device="cuda")
    rhoc[0, at[:, None, None], at[None, :, None], at[None, None, :]] = n
    idx = rhoc.long().sum(3).reshape(-1).cumsum(0).reshape(1, g.nte, g.nte).contiguous()
    return g, rhoc, idx, 8 * n


def _numbered(n):
    import torch
    i = torch.arange(n, dtype=torch.int32, device="cuda")
    return torch.stack([(i & 0xfffff).float(), (i >> 20).float(), -(i & 0xfffff).float()], 1)


def test_halo_velocities_and_positions_of_more_than_2_31_slots():
    """2^31 + 40 slots: the halo copies' velocities are their particles', every
    position is its code decoded in the corner cell."""
    import torch
    from cube2_amd.drift import refresh_halo_velocities, slot_positions_device
    n = (1 << 28) + 5
    g, rhoc, idx, slots = _corner_image(n)
    print(f"{slots} slots", flush=True)
    vel = _numbered(n)
    vp = torch.full((slots, 3), -7.0, device="cuda")
    vp[:n] = vel  # (the first of the 8 cells is the physical one)
    refresh_halo_velocities(rhoc, idx, vp, slots, g)
    for k in range(8):
        assert torch.equal(vp[k * n:(k + 1) * n], vel), k
    del vp, vel
    xp = torch.randint(-32768, 32768, (slots, 3), dtype=torch.int16, device="cuda")
    pos = slot_positions_device(rhoc, idx, xp, slots, g)
    for k in range(32):
        a, b = slots * k // 32, slots * (k + 1) // 32
        want = ((xp[a:b].int() & 0xffff).double() + 0.5) / 65536.0 * g.ratio_cs
        assert torch.equal(pos[a:b], want), k


def test_drift_of_nearly_2_31_slots():
    """2^31 - 8 slots, a step of zero: the corner cell's particles stay."""
    import ctypes as C

    import torch
    from cube2_amd import _lib
    n = (1 << 28) - 1
    g, rhoc, idx, slots = _corner_image(n)
    print(f"drift of {slots} slots", flush=True)
    _lib.set_params(g)
    vp = _numbered(n).repeat(8, 1)
    xp = torch.randint(-32768, 32768, (n, 3), dtype=torch.int16, device="cuda").repeat(8, 1)
    r, i = torch.empty_like(rhoc), torch.empty_like(idx)
    x = torch.empty((n, 3), dtype=torch.int16, device="cuda")
    v = torch.empty((n, 3), device="cuda")
    kept = C.c_int64(0)
    _lib.check(_lib.lib().cube2_drift_dev(rhoc.data_ptr(), idx.data_ptr(), xp.data_ptr(), vp.data_ptr(),
                                          slots, 0.0, 1.0, r.data_ptr(), i.data_ptr(), x.data_ptr(),
                                          v.data_ptr(), n, C.byref(kept)))
    assert kept.value == n == int(r[0, g.ncb, g.ncb, g.ncb]) == int(r.sum())
    assert torch.equal(x, xp[:n]) and torch.equal(v, vp[:n])
