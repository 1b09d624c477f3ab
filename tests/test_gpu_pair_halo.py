"""The pair form with a ghost copy list, whose launches read a ghost's source
in its place from the third on: chains of runs of every length around that
change, sources of every kind (active and inactive points, none), ghosts that
start away from their source, bit for bit against the oracle after every run."""
import numpy as np
import pytest

from gpu_common import assert_state_bitexact, fetch_state, make_engine, oracle_params, synthetic_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ice,chain", [
    (45, 37, 0.7, (1, 2, 3, 4, 5, 6, 7, 8, 9)),
    (45, 37, 0.3, (13, 4, 6)),
    (260, 200, 0.8, (7, 8)),
])
def test_chain(gpu, nx, ny, ice, chain):
    st = synthetic_state(nx, ny, seed=77, ice_prob=ice)
    r = np.random.default_rng(9)
    ghosts = np.arange(st.na + 1, st.navel + 1, dtype=np.int32)
    dst = r.choice(ghosts, size=3 * ghosts.size // 4, replace=False).astype(np.int32)
    src = r.integers(0, st.na + 1, size=dst.size).astype(np.int32)   # 0 = fill with zero
    for n in ("uvel", "vvel"):
        st.f[n][st.na:] = 0.05 * r.standard_normal(st.navel - st.na)
    lib, p = oracle_params(st, 120)
    want = st.copy()
    with make_engine(st, 120, "fused") as eng:
        eng.set_fused_depth(2)
        eng.set_halo(dst, src)
        assert eng.get_fused_depth()["active"]
        for nsub in chain:
            eng.run(nsub)
            lib.run(p, want, nsub, halo=(dst, src))
            assert_state_bitexact(fetch_state(eng, st), want)
