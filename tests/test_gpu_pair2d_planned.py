"""The 2D path's pair form, planned beside a run of 2000 subcycles and then
given fresh fields: against the plain form on the rows of test_gpu_pair2d.py,
bit for bit on every array, and against the reference's own output files.
That these runs take the pair form, which no result shows, is what
test_pair2d_rule.py holds."""
import numpy as np
import pytest

import evp1d
from evp1d import synth
from gpu_common import golden_cases_v0, load_golden_v0
from oracle import oracle as O
from test_gpu_pair2d import _random_halo, _random_lists

pytestmark = pytest.mark.gpu


def _everywhere(st, seed=4):
    """Values of the ocean in the dry cells too: the lists below take any cell,
    and one dry U cell's 0/0 would soon make NaN of all that is compared."""
    r = np.random.default_rng(seed)
    for n in evp1d.FIELDS2D[:42]:
        a = st.f[n]
        some = a[a != 0.0]
        if some.size:
            a[a == 0.0] = r.choice(some, (a == 0.0).sum())
    return st


def _fields(eng, st):
    for n in evp1d.FIELDS2D[:42]:
        eng.set_field(n, st.f[n])


@pytest.mark.parametrize("nx,ny,nblocks,share,halo_u,nsub", [
    (12, 9, 1, 1.0, False, 4),
    (70, 45, 1, 0.6, False, 7),
    (70, 45, 3, 0.8, False, 9),
    (60, 33, 4, 0.3, False, 4),
    (40, 30, 2, 1.0, True, 6),
    (250, 190, 2, 1.0, False, 5),
    (700, 480, 1, 1.0, False, 4),
    (600, 400, 1, 1.0, False, 5),
])
def test_pair_form_equals_plain_form(gpu, nx, ny, nblocks, share, halo_u, nsub):
    st = _everywhere(O.pack_v0(synth.make_grid(nx, ny, 61, land_frac=0.1), nblocks))
    got = []
    for mode in ("plain", "fused"):
        r = np.random.default_rng(99)
        with evp1d.Engine2D(st.nxb, st.nyb, st.nblocks, evp1d.set_evp_parameters(120)) as eng:
            eng.load_state(st)
            _random_lists(eng, st, r, share, halo_u)
            if nblocks > 1:
                eng.set_halo(*_random_halo(eng, r))
            eng.set_mode(mode)
            eng.run(2000)
            got.append([eng.get_field(n) for n in evp1d.FIELDS2D])
            _fields(eng, st)
            eng.run(nsub)
            eng.run(4)
            got[-1] += [eng.get_field(n) for n in evp1d.FIELDS2D]
    for k, (a, b) in enumerate(zip(*got)):
        same = (a.view(np.uint64) == b.view(np.uint64)) | (np.isnan(a) & np.isnan(b))
        assert same.all(), f"{evp1d.FIELDS2D[k % len(evp1d.FIELDS2D)]}: {(~same).sum()} of {a.size} values differ"
    assert all(bool(np.isfinite(a).all()) for a in got[1][len(evp1d.FIELDS2D):])


@pytest.mark.parametrize("case", golden_cases_v0())
def test_golden_outputs(gpu, case):
    st, ndte, want_stress, want_stepu = load_golden_v0(case)
    p = evp1d.set_evp_parameters(ndte)
    for k in ("capping", "e_factor", "epp2i"):
        setattr(p, k, st.scalars[k])
    with evp1d.Engine2D(st.nxb, st.nyb, st.nblocks, p) as eng:
        eng.load_state(st)
        eng.run(2000)
        _fields(eng, st)
        eng.run(ndte)
        got = st.copy()
        for n in O.V0_FIELDS:
            got.f[n][:] = eng.get_field(n)
    assert O.output_bytes_v0(got) == (want_stress, want_stepu)
