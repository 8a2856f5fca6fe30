"""The autotuner's search over a stand-in for the kick's time: which pair kernel
runs is settled before its launch shapes, and both kernels' useful shapes are
among the candidates (the pairs-once kernel's wavefronts take parts from
counters, so that its grids are at most what is resident; the ordered kernel's
are many times that)."""
from __future__ import annotations

import pytest

from cube2_amd import _lib, autotune

NAMES = {v: k for k, v in _lib.TUNE_NAMES.items()}


class Kick:
    def kick(self, *args):
        pass


@pytest.mark.parametrize("once,best", [(1.0, {"pp_overlap_blocks": 2, "pp_blocks_per_cu": 4}),
                                       (1.0, {"pp_overlap_blocks": 6, "pp_blocks_per_cu": 8}),
                                       (1.0, {"pp_overlap_blocks": 4}),
                                       (9.0, {"pp_overlap_blocks": 96, "pp_blocks_per_cu": 24}),
                                       (9.0, {"pp_overlap_blocks": 32, "pp_blocks_per_cu": 128})])
def test_the_tuner_finds_the_shapes_of_the_kernel_it_chose(monkeypatch, once, best):
    """Pairs once takes `once`, ordered 5; each kernel loses a quarter without its
    best shapes and has no use for the other's."""
    state = {}
    monkeypatch.setattr(_lib, "set_tuning", lambda key, v: state.__setitem__(NAMES[key], v))

    def time_kick(kick, mass, a_mid, dt, reps):
        ordered = state.get("pp_newton") == 2
        t = 5.0 if ordered else once
        mine = best if ordered == (once > 5.0) else {}
        return t * 1.25 ** sum(state.get(n, 0) != v for n, v in mine.items())

    monkeypatch.setattr(autotune, "_time_kick", time_kick)
    chosen = autotune.autotune(Kick(), 1.0, 1.0, 1.0)["chosen"]
    assert chosen["pp_newton"] == (2 if once > 5.0 else 0)
    assert {n: chosen[n] for n in best} == best
    assert chosen == {n: state[n] for n in chosen}  # left set in the library
