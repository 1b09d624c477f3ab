"""When the 2D path plans the pair form and what its runs launch (CPU:
tests/fake_hip.py): beside a run, when the subcycles on the same lists pay for
it, never inside a getter."""
import numpy as np
import pytest

import evp1d
from evp1d import synth
from fake_hip import bound, build_fake, fake, fake_lib  # noqa: F401
from oracle import oracle as O
from test_gpu_pair2d import _random_halo, _random_lists


def _engine(nx=70, ny=45, nblocks=2, fma=False):
    st = O.pack_v0(synth.make_grid(nx, ny, 61, land_frac=0.1), nblocks)
    eng = evp1d.Engine2D(st.nxb, st.nyb, st.nblocks, evp1d.set_evp_parameters(120, fma=fma), fma=fma)
    eng.load_state(st)
    return eng, st


def _run(eng, fake, nsub):
    """(subcycles run one per launch, two per launch) by eng.run(nsub), checked for their sum and order."""
    fake.launches()
    eng.run(nsub)
    form = [n.split("<")[0] for n in fake.kernels() if n.startswith(("k2_fused", "k_pair"))]
    one, two = form.count("k2_fused"), 2 * form.count("k_pair")
    assert one + two == nsub and form == sorted(form)
    return one, two


def test_short_runs_do_not_pay_for_a_plan(fake):
    eng, st = _engine()
    with eng:
        done = 0
        while True:
            want = done > 0 and done + 12 >= 4 * (500 - 12)
            assert _run(eng, fake, 12) == (12, 0)       # the run beside which the plan is made is done by then
            done += 12
            if want:
                break
        assert done > 1900
        assert _run(eng, fake, 12) == (0, 12)
        assert _run(eng, fake, 13) == (1, 12)
        assert _run(eng, fake, 3) == (3, 0)
        eng.load_state(st)                               # new lists
        assert _run(eng, fake, 12) == (12, 0)


@pytest.mark.parametrize("nsub", [1000, 1001])
def test_plan_beside_a_second_run(fake, nsub):
    eng, _ = _engine()
    with eng:
        assert _run(eng, fake, nsub) == (nsub, 0)
        one = 500 + nsub % 2
        assert _run(eng, fake, nsub) == (one, nsub - one)
        assert _run(eng, fake, nsub) == (nsub % 2, nsub - nsub % 2)


def test_plan_beside_a_long_first_run(fake):
    eng, _ = _engine()
    with eng:
        assert _run(eng, fake, 1999) == (1999, 0)
    eng, _ = _engine()
    with eng:
        assert _run(eng, fake, 2000) == (500, 1500)


@pytest.mark.parametrize("nsub", [12, 1000])
def test_getter_between_runs(fake, nsub):
    """It neither plans nor keeps the plan's form from the runs after it."""
    runs = []
    for ask in (False, True):
        eng, _ = _engine()
        with eng:
            eng.set_cache_hints(1)
            runs.append([])
            for _ in range(3):
                runs[-1].append(_run(eng, fake, nsub))
                if ask:
                    live = fake.live()
                    assert eng.get_cache_hints() == {"hints": 1, "active": True}
                    assert fake.live() == live
    assert runs[0] == runs[1]


def test_contracted_build_keeps_one_form(tmp_path):
    with bound(build_fake(tmp_path, True), True) as fake:
        eng, _ = _engine(fma=True)
        with eng:
            assert _run(eng, fake, 2000) == (2000, 0)
            assert _run(eng, fake, 1000) == (1000, 0)


# the rows of test_gpu_pair2d.py and test_gpu_pair2d_planned.py: the tiles' size, or None
@pytest.mark.parametrize("nx,ny,nblocks,share,halo_u,tile,threads", [
    (12, 9, 1, 1.0, False, (15, 11), 256),
    (70, 45, 1, 0.6, False, (15, 11), 256),
    (70, 45, 3, 0.8, False, (15, 11), 256),
    (60, 33, 4, 0.3, False, (15, 11), 256),
    (40, 30, 2, 1.0, True, None, 0),                # stepu writes a halo cell
    (250, 190, 2, 1.0, False, (22, 16), 512),
    (700, 480, 1, 1.0, False, (31, 13), 512),
    (600, 400, 1, 1.0, False, (31, 15), 512),       # crowded in 31x17
])
def test_rows_of_the_gpu_tests(fake, nx, ny, nblocks, share, halo_u, tile, threads):
    eng, st = _engine(nx, ny, nblocks)
    r = np.random.default_rng(99)
    with eng:
        _random_lists(eng, st, r, share, halo_u)
        if nblocks > 1:
            eng.set_halo(*_random_halo(eng, r))
        if tile is None:
            assert _run(eng, fake, 2000) == (2000, 0)
            return
        assert _run(eng, fake, 2000) == (500, 1500)
        fake.launches()
        eng.run(5)
        pair = [x for x in fake.launches() if x[0].startswith("k_pair")]
    assert len(pair) == 2 and {x[2] for x in pair} == {threads}
    copies = "true" if nblocks > 1 else "false"
    assert {x[0] for x in pair} == {f"k_pair<{threads}, true, false, {copies}, false>"}
    # blocks stand side by side, one column apart; the lists leave out the first and last cells
    cells = np.zeros((nblocks * (st.nxb + 1), st.nyb), bool)
    for b in range(nblocks):
        cells[b * (st.nxb + 1) + 1:b * (st.nxb + 1) + st.nxb, 1:st.nyb] = True
    i, j = np.nonzero(cells)
    tiles = len(set(zip(i // tile[0], j // tile[1])))
    assert {x[1] for x in pair} <= ({tiles} if share == 1.0 else set(range(1, tiles + 1)))
