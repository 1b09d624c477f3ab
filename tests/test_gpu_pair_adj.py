"""The gradient's reverse sweep in the pair form (two subcycles per launch)
against one kernel per point class (fused depth 1), bit for bit on the loss
and the four gradients: every remainder of the number of subcycles, tiles of
every workgroup size, both cache hint settings, the whole trajectory and
checkpointed units of odd and even length."""
import numpy as np
import pytest

from gpu_common import make_engine, synthetic_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ice,nsub,nsnap,hints", [
    (1, 1, 1.0, 3, 0, -1),
    (40, 30, 0.7, 1, 0, -1),
    (40, 30, 0.7, 2, 0, -1),
    (40, 30, 0.7, 3, 0, 1),
    (40, 30, 0.7, 4, 0, 0),
    (70, 50, 0.4, 9, 3, -1),         # units of 3
    (70, 50, 1.0, 16, 4, 1),         # units of 4, the sweep's stresses packed from the stored states
    (70, 50, 0.7, 10, 4, -1),        # units of 3 made 4: 4, 4, 2
    (352, 257, 1.0, 5, 0, -1),       # 1024 threads
    (497, 304, 0.7, 6, 0, 1),        # 31x15
    (620, 480, 0.7, 5, 0, 0),        # 31x19, 512 threads
])
def test_pair_reverse_equals_single_kernels(gpu, nx, ny, ice, nsub, nsnap, hints):
    st = synthetic_state(nx, ny, seed=17, land_frac=0.1 if nx > 1 else 0.0, ice_prob=ice)
    r = np.random.default_rng(3)
    ut, vt = 0.1 * r.standard_normal(st.na), 0.1 * r.standard_normal(st.na)
    got, t = [], None
    for depth in (2, 1):
        with make_engine(st, nsub) as eng:
            eng.set_fused_depth(depth)
            eng.set_cache_hints(hints)
            t = t or eng.get_tiling()
            eng.set_tiling(t["tile_w"], t["tile_h"], t["block"])   # one slot order: the loss is summed in it
            assert eng.get_fused_depth()["active"] == (depth == 2)
            got.append(eng.adjoint_run(nsub, ut, vt, nsnap=nsnap))
    for n in ("loss", "strength", "cdn_ocn", "forcex", "forcey"):
        a, b = (np.atleast_1d(np.asarray(g[n], np.float64)) for g in got)
        assert np.array_equal(a, b), f"{n}: {(a != b).sum()} of {a.size} values differ"
