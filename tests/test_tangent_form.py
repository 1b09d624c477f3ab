"""The form that each row of test_gpu_fused_tangent.py takes (CPU:
tests/fake_hip.py): no result of those rows shows it."""
import numpy as np
import pytest

from fake_hip import fake, fake_lib  # noqa: F401
from gpu_common import make_engine, synthetic_state


@pytest.mark.parametrize("nx,ny,ice,nsub,tile,want", [
    (1, 1, 1.0, 1, None, "k_fused_tl<256>"),
    (50, 40, 0.7, 5, None, "k_fused_tl<256>"),
    (300, 200, 0.7, 4, None, "k_fused_tl<512>"),
    (352, 257, 1.0, 3, None, "k_fused_tl<512>"),
    (120, 90, 0.5, 6, (64, 8, 256), "k_fused_tl<512>"),
    (120, 90, 0.8, 5, (64, 32, 512), "k_stress_tl"),
])
def test_form(fake, nx, ny, ice, nsub, tile, want):
    st = synthetic_state(nx, ny, seed=23, land_frac=0.1 if nx > 1 else 0.0, ice_prob=ice)
    z = np.zeros(st.na)
    with make_engine(st, nsub) as eng:
        if tile:
            eng.set_tiling(*tile)
        fake.launches()
        eng.tangent_run(nsub, z, z)
        got = fake.launches()
    forms = [x for x in got if x[0].startswith(("k_fused_tl", "k_stress_tl"))]
    assert [x[0] for x in forms] == nsub * [want]
    if tile == (64, 8, 256):      # more entries of 8 pairs than the 512 threads
        assert forms[0][3] > 512 * 128
