"""The fused tangent (one tile per workgroup, values and derivatives side by
side) over its workgroup sizes and over tiles whose tables do not fit (the
unfused form): the state it leaves is the forward's bit for bit against the
oracle, and its derivative is the inner product of the gradient with the
direction, to the 1e-10 that the dot-product test of the two modes holds."""
import numpy as np
import pytest

from gpu_common import assert_state_bitexact, fetch_state, make_engine, oracle_params, synthetic_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ice,nsub,tile", [
    (1, 1, 1.0, 1, None),
    (50, 40, 0.7, 5, None),             # 15x11: 256 threads
    (300, 200, 0.7, 4, None),           # 22x16: 512 threads
    (352, 257, 1.0, 3, None),           # 31x19, more entries than threads
    (120, 90, 0.5, 6, (64, 8, 256)),    # more entries than threads, 512
    (120, 90, 0.8, 5, (64, 32, 512)),   # tables beyond LDS: unfused
])
def test_tangent_state_and_derivative(gpu, nx, ny, ice, nsub, tile):
    st = synthetic_state(nx, ny, seed=23, land_frac=0.1 if nx > 1 else 0.0, ice_prob=ice)
    r = np.random.default_rng(8)
    ut, vt = 0.1 * r.standard_normal(st.na), 0.1 * r.standard_normal(st.na)
    d = {n: r.random(st.na) * np.abs(st.f[n]) for n in ("strength", "cdn_ocn", "forcexU", "forceyU")}
    with make_engine(st, nsub) as eng:
        if tile:
            eng.set_tiling(*tile)
        loss, along = eng.tangent_run(nsub, ut, vt, d["strength"], d["cdn_ocn"], d["forcexU"], d["forceyU"])
        got = fetch_state(eng, st)
    lib, p = oracle_params(st, nsub)
    want = st.copy()
    lib.run(p, want, nsub)
    assert_state_bitexact(got, want)
    with make_engine(st, nsub) as eng:
        g = eng.adjoint_run(nsub, ut, vt)
    parts = (np.dot(g["strength"], d["strength"]), np.dot(g["cdn_ocn"], d["cdn_ocn"]),
             np.dot(g["forcex"], d["forcexU"]), np.dot(g["forcey"], d["forceyU"]))
    assert abs(loss - g["loss"]) <= 1e-12 * abs(g["loss"])
    assert abs(along - sum(parts)) <= 1e-10 * max(map(abs, parts))
