"""The tile that the library chooses for the pair form, at the edges of its
ladder (one tile per CU: 15x11, 22x16, 26x16, 31x15, 31x17, 31x19; two per CU:
22x16, 26x16, 31x15, 31x17, 31x19; four: 31x13; 31x19; 31x15 where contiguous
ice crowds the larger ones): the choice, and the state after a run bit for bit
against the oracle."""
import pytest

from gpu_common import assert_state_bitexact, fetch_state, make_engine, oracle_params, synthetic_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ice,tile,threads", [
    (1, 1, 1.0, (15, 11), 256),
    (240, 176, 1.0, (15, 11), 256),     # 16 x 16 tiles: 256
    (241, 176, 1.0, (22, 16), 512),
    (352, 256, 0.7, (22, 16), 512),     # 16 x 16 tiles of 22x16
    (352, 257, 1.0, (26, 16), 512),     # 14 x 17 of 26x16
    (496, 240, 0.7, (31, 15), 512),     # 16 x 16 of 31x15
    (496, 272, 1.0, (31, 17), 1024),    # 16 x 16 of 31x17, 576 level-2 points each
    (496, 304, 1.0, (31, 19), 1024),    # 16 x 16 of 31x19
    (497, 304, 0.7, (22, 16), 512),     # 17 x 16 of 31x19; 23 x 19 of 22x16
    (520, 400, 0.7, (26, 16), 512),     # 20 x 25 of 26x16
    (620, 375, 0.7, (31, 15), 512),     # 20 x 25 of 31x15
    (620, 425, 0.7, (31, 17), 512),     # 20 x 25 of 31x17
    (620, 475, 0.7, (31, 19), 512),     # 20 x 25 of 31x19
    (620, 480, 0.7, (31, 13), 512),     # 20 x 26 of 31x19
    (620, 480, 1.0, (31, 13), 512),
    (620, 425, 1.0, (31, 15), 512),     # 20 x 25 of 31x17, crowded
    (1240, 336, 0.7, (31, 19), 512),    # 40 x 26 of 31x13: more than 1024
    (1240, 336, 1.0, (31, 15), 512),    # 640 level-2 points in a 31x19 tile
])
def test_chosen_tile(gpu, nx, ny, ice, tile, threads):
    st = synthetic_state(nx, ny, seed=5, land_frac=0.0, ice_prob=ice)
    nsub = 4
    with make_engine(st, nsub) as eng:
        t, d = eng.get_tiling(), eng.get_fused_depth()
        assert (t["tile_w"], t["tile_h"]) == tile and d["active"] and d["block"] == threads
        eng.run(nsub)
        got = fetch_state(eng, st)
    lib, p = oracle_params(st, nsub)
    want = st.copy()
    lib.run(p, want, nsub)
    assert_state_bitexact(got, want)
