"""The 2D path's pair form (two subcycles per launch) against its plain form
(stress then stepu, as the reference runs them), bit for bit on every array:
cell lists in any order that no ice mask would give, halo copies from other
blocks into sides and corners, zero fills, copies of filled cells, a halo cell
that stepu writes (the pair form then steps aside), odd and even runs, tiles
of every rung."""
import numpy as np
import pytest

import evp1d
from evp1d import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _random_lists(eng, st, rng, share, halo_u):
    nxb, nyb, nb = eng.shape
    for b in range(nb):
        t = [(i, j) for i in range(2, nxb + 1) for j in range(2, nyb + 1) if rng.random() < share]
        u = [(i, j) for i in range(2, nxb) for j in range(2, nyb) if rng.random() < share]
        if halo_u and b == 0:
            u.append((1, 2))
        rng.shuffle(t)
        rng.shuffle(u)
        t, u = np.array(t, np.int32).reshape(-1, 2), np.array(u, np.int32).reshape(-1, 2)
        eng.set_cells(b + 1, t[:, 0], t[:, 1], u[:, 0], u[:, 1])


def _random_halo(eng, rng):
    nxb, nyb, nb = eng.shape
    rim = [(i, j, b) for b in range(1, nb + 1) for i in range(1, nxb + 1) for j in range(1, nyb + 1)
           if i in (1, nxb) or j in (1, nyb)]
    dst = [c for c in rim if rng.random() < 0.7]
    left = [c for c in rim if c not in set(dst)]          # filled with zero, and copied as zero
    src = [left[rng.integers(len(left))] if left and rng.random() < 0.1 else
           (0, 0, 0) if rng.random() < 0.1 else
           (int(rng.integers(2, nxb)), int(rng.integers(2, nyb)), int(rng.integers(1, nb + 1))) for _ in dst]
    one = np.ones(nb, np.int32)
    return 2 * one, 2 * one, (nxb - 1) * one, (nyb - 1) * one, np.array(src, np.int32).T, np.array(dst, np.int32).T


@pytest.mark.parametrize("nx,ny,nblocks,share,halo_u,nsub", [
    (12, 9, 1, 1.0, False, 4),
    (70, 45, 1, 0.6, False, 7),
    (70, 45, 3, 0.8, False, 9),
    (60, 33, 4, 0.3, False, 4),
    (40, 30, 2, 1.0, True, 6),
    (250, 190, 2, 1.0, False, 5),     # more than one 15x11 tile per CU: 22x16
    (700, 480, 1, 1.0, False, 4),     # a crowded 31x19 tile: 31x15
])
def test_pair_form_equals_plain_form(gpu, nx, ny, nblocks, share, halo_u, nsub):
    st = O.pack_v0(synth.make_grid(nx, ny, 61, land_frac=0.1), nblocks)
    got = []
    for mode in ("plain", "fused"):
        r = np.random.default_rng(99)
        with evp1d.Engine2D(st.nxb, st.nyb, st.nblocks, evp1d.set_evp_parameters(120)) as eng:
            eng.load_state(st)
            _random_lists(eng, st, r, share, halo_u)
            if nblocks > 1:
                eng.set_halo(*_random_halo(eng, r))
            eng.set_mode(mode)
            eng.run(2)           # lists are planned for the pair form at their second run
            eng.run(nsub)
            eng.run(4)
            got.append({n: eng.get_field(n) for n in evp1d.FIELDS2D})
    for n in evp1d.FIELDS2D:
        a, b = got[0][n], got[1][n]
        same = (a.view(np.uint64) == b.view(np.uint64)) | (np.isnan(a) & np.isnan(b))
        assert same.all(), f"{n}: {(~same).sum()} of {a.size} values differ"
