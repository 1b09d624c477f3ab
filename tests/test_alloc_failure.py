"""Allocations that fail inside a call (CPU: tests/fake_hip.py): the call says
so or takes the form that needs less, and the same call made again, with the
memory there, launches what it would have launched."""
import numpy as np
import pytest

import evp1d
from evp1d import synth
from fake_hip import fake, fake_lib  # noqa: F401
from gpu_common import make_engine, synthetic_state
from oracle import oracle as O


def _engine2d():
    st = O.pack_v0(synth.make_grid(70, 45, 61, land_frac=0.1), 3)
    eng = evp1d.Engine2D(st.nxb, st.nyb, st.nblocks, evp1d.set_evp_parameters(120))
    eng.load_state(st)
    return eng


# 4: one subcycle per launch; 2000 and more: the pair form, for which three
# failures leave the one-subcycle tables short of memory too
@pytest.mark.parametrize("nsub,count", [(4, 1), (2000, 1), (2001, 3)])
def test_2d_run_after_a_failed_one(fake, nsub, count):
    with _engine2d() as eng:
        fake.launches()
        eng.run(nsub)
        want = fake.launches()
    for after in range(40):
        with _engine2d() as eng:
            fake.launches()
            fake.fail(after, count)
            try:
                eng.run(nsub)
                failed = False
            except evp1d.Evp1dError as e:
                assert e.code in (3, 4)
                failed = True
            fake.no_fail()
            got = fake.launches()
            if not failed:
                assert any("k2_fused" in n or "k_pair" in n for n, *_ in got), after
                if got == want:
                    break                  # beyond the run's last allocation
                continue                   # the form that needs less
            assert got == [], after
            eng.run(nsub)
            assert any("k2_fused" in n or "k_pair" in n for n, *_ in fake.launches()), after
    else:
        assert False, "more allocations than tried"


def _engine1d():
    st = synthetic_state(150, 110, 5, ice_prob=0.7)
    return make_engine(st, 120)


def test_1d_after_a_failed_plan(fake):
    """The second run plans the tiles.  Where that fails the points may have a
    new order already: the neighbour lists follow it before anything runs."""
    seen = set()
    for after in range(60):
        with _engine1d() as eng:
            eng.run(4)                # class order
            fake.launches()
            fake.fail(after)
            try:
                eng.run(4)
            except evp1d.Evp1dError as e:
                assert e.code in (3, 4)
                fake.no_fail()
                eng.stress()
                got = fake.kernels()
                assert got[-1].startswith("k_stress"), after
                moved = [k for k, n in enumerate(got) if n == "k_permute_pair"]
                assert not moved or "k_idx_to_slots" in got[moved[-1]:], after
                seen.add(bool(moved))
                eng.run(4)
                assert any(n.startswith(("k_pair", "k_stepu")) for n in fake.kernels()), after
            else:
                break
    assert True in seen


def test_gradient_and_tangent_take_the_form_that_needs_less(fake):
    st = synthetic_state(150, 110, 5, ice_prob=0.7)
    z = np.zeros(st.na)
    for call, fast, less in (("adjoint_run", "k_pair_adj", "k_stress_adj"), ("tangent_run", "k_fused_tl", "k_stress_tl")):
        forms = []
        for after in range(60):
            with _engine1d() as eng:
                eng.run(500)          # planned
                fake.launches()
                fake.fail(after)
                args = (6, z, z) if call == "adjoint_run" else (6, z, z, z, z, z, z)
                try:
                    getattr(eng, call)(*args)
                    failed = False
                except evp1d.Evp1dError as e:
                    assert e.code in (3, 4)
                    failed = True
                fake.no_fail()
                got = fake.kernels()
                if not failed:
                    forms.append("fast" if any(n.startswith(fast) for n in got) else "less")
                    assert forms[-1] == "fast" or any(n.startswith(less) for n in got), (call, after)
                    if forms[-1] == "fast":
                        break
                    continue
                getattr(eng, call)(*args)
                assert any(n.startswith(fast) for n in fake.kernels()), (call, after)
        assert "less" in forms and forms[-1] == "fast", (call, forms)
