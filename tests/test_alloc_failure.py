"""Allocations that fail inside a call (CPU: tests/fake_hip.py): the call says
so or takes the form that needs less, and the same call made again, with the
memory there, launches what it would have launched."""
import pytest

import evp1d
from evp1d import synth
from fake_hip import fake, fake_lib  # noqa: F401
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
