"""The slot-parallel kernels at the largest slot counts: every slot is written
where the count ends within a block of 2^31.  Copies: bit-exact."""
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
    i = torch.arange(n, dtype=torch.int32, device="cuda")
    vel = torch.stack([(i & 0xfffff).float(), (i >> 20).float(), -(i & 0xfffff).float()], 1)
    del i
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
