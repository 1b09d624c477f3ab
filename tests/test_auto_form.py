"""The form that evp1d_run takes in AUTO mode (CPU: tests/fake_hip.py): the
first short run with new skip flags goes over the points in class order;
tiles, orders and depths that were asked for, a copy list that changes and
later runs take the tiles."""
import ctypes

import numpy as np
import pytest

from fake_hip import fake, fake_lib  # noqa: F401
from gpu_common import make_engine, synthetic_state


@pytest.fixture
def st():
    return synthetic_state(150, 110, 5, ice_prob=0.7)


def _form(fake):
    """"class order", "pairs" or "tiles" (one subcycle each) of the last run."""
    names = {n.split("<")[0] for n in fake.kernels()}
    return ("pairs" if "k_pair" in names else "tiles" if "k_fused" in names else
            "class order" if "k_stress" in names else names)


def _run(eng, fake, nsub=120):
    fake.launches()
    eng.run(nsub)
    return _form(fake)


def test_new_flags(fake, st):
    with make_engine(st, 120) as eng:
        assert _run(eng, fake) == "class order"
        assert _run(eng, fake) == "pairs"
        flags = st.skipT.copy()
        flags[:50] = 1
        eng.set_skip("skipT", flags)
        assert _run(eng, fake) == "class order"
        eng.set_skip("skipT", flags)                   # the same ones
        assert _run(eng, fake) == "pairs"
        eng.set_skip("skipT", st.skipT)
        assert _run(eng, fake, 500) == "pairs"         # long enough
        eng.set_skip("skipT", flags)
        eng.loss(np.zeros(st.na), np.zeros(st.na))     # a new layout, but no run
        assert _run(eng, fake) == "class order"


@pytest.mark.parametrize("ask", ["tiling", "order", "depth", "autotune", "tiling before the flags"])
def test_settings_asked_for_are_what_the_next_run_takes(fake, st, ask):
    with make_engine(st, 120) as eng:
        if ask == "tiling before the flags":
            eng.set_tiling(20, 10, 256)
            eng.set_skip("skipT", 1 - st.skipT)
            eng.set_skip("skipT", st.skipT)
        if ask == "tiling":
            eng.set_tiling(20, 10, 256)
        if ask == "order":
            eng.set_tile_order(1)
        if ask == "depth":
            eng.set_fused_depth(1)
        if ask == "autotune":
            us = ctypes.c_float()
            assert eng.L.evp1d_autotune_fused(eng.h, 4, ctypes.byref(us)) == 0
        assert _run(eng, fake, 12) == ("tiles" if ask in ("depth", "autotune") else "pairs")
        eng.set_skip("skipT", 1 - st.skipT)            # later flags are new flags again
        assert _run(eng, fake, 12) == "class order"


@pytest.mark.parametrize("setting", ["tiling", "order", "depth", "halo"])
def test_settings_that_change_later_bring_no_class_order_back(fake, st, setting):
    with make_engine(st, 120) as eng:
        eng.run(12)
        eng.run(12)
        if setting == "tiling":
            eng.set_tiling(20, 10, 256)
        if setting == "order":
            eng.set_tile_order(1)
        if setting == "depth":
            eng.set_fused_depth(1)
        if setting == "halo":
            eng.set_halo(np.array([st.na + 1], np.int32), np.array([1], np.int32))
        assert _run(eng, fake, 12) == ("tiles" if setting == "depth" else "pairs")


def test_tiles_planned_by_a_getter_are_what_the_first_run_takes(fake, st):
    with make_engine(st, 120) as eng:
        assert eng.get_fused_depth()["active"]
        assert _run(eng, fake) == "pairs"


def _sets(eng, fake, st, runs, sets):
    """Forms of the runs of each of `sets` model steps, each with flags of its own."""
    forms = []
    for k in range(sets):
        flags = st.skipT.copy()
        flags[k] ^= 1
        eng.set_skip("skipT", flags)
        forms.append([_run(eng, fake, n) for n in runs])
    return forms


def test_steps_of_several_short_runs(fake, st):
    with make_engine(st, 120) as eng:
        once, never = ["class order", "pairs"], ["class order", "class order"]
        assert _sets(eng, fake, st, [120, 120], 5) == [once, once, never, never, never]
        assert [_run(eng, fake, 120) for _ in range(4)] == ["class order", "class order", "pairs", "pairs"]
        # a set that had enough for a plan: the second run of the next one plans again
        assert _sets(eng, fake, st, [120, 120], 1) == [once]


def test_steps_of_several_runs_long_enough_together(fake, st):
    with make_engine(st, 120) as eng:
        second, first = ["class order", "pairs"], ["pairs", "pairs"]
        assert _sets(eng, fake, st, [300, 200], 4) == [second, second, first, first]
        assert _sets(eng, fake, st, [120, 120], 2) == [first, second]
