"""evp1d_run without tiles: the first short run with new skip flags goes over
the points in class order, later or long ones over tiles.  A chain of runs
and changing flags (none active, all active, few) through that change of slot
order, bit for bit against the oracle after every run."""
import numpy as np
import pytest

from gpu_common import assert_state_bitexact, fetch_state, make_engine, oracle_params, synthetic_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,chain", [
    (1, 1, [(1.0, 3), (1.0, 4)]),
    (60, 45, [(0.7, 5), (0.7, 6), (0.2, 1), (0.9, 4), (0.9, 500), (0.0, 3), (0.5, 3), (0.5, 2), (1.0, 5)]),
    (60, 45, [(0.7, 499), (0.3, 500), (0.3, 7)]),
    (330, 260, [(0.6, 4), (0.8, 7), (0.8, 5)]),       # more than one chunk of the parallel class order
])
def test_chain_of_runs_and_flags(gpu, nx, ny, chain):
    st = synthetic_state(nx, ny, seed=12, land_frac=0.1 if nx > 1 else 0.0, ice_prob=1.0)
    lib, p = oracle_params(st, 120)
    r = np.random.default_rng(5)
    share, want = None, st.copy()
    with make_engine(st, 120) as eng:
        for s, nsub in chain:
            if s != share:
                share = s
                want.skipT[:] = r.random(st.na) >= s
                want.skipU[:] = r.random(st.na) >= s
                eng.set_skip("skipT", want.skipT)
                eng.set_skip("skipU", want.skipU)
            eng.run(nsub)
            lib.run(p, want, nsub)
            assert_state_bitexact(fetch_state(eng, st), want)
        assert eng.get_fused_depth()["active"] == bool((want.skipT == 0).any())


def test_contracted_build_keeps_one_form(gpu):
    """libevp1d_fma.so rounds by form: its first run takes the form that the
    later ones take."""
    st = synthetic_state(60, 45, seed=12, ice_prob=0.7)
    got = []
    for planned in (False, True):
        with make_engine(st, 120, fma=True) as eng:
            if planned:
                assert eng.get_fused_depth()["active"]   # plans the tiles
            eng.run(6)
            eng.run(7)
            got.append(fetch_state(eng, st))
    assert_state_bitexact(got[0], got[1])
