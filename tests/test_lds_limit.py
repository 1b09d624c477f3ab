"""The LDS that a kernel may use is an attribute of the kernel, not of a
handle (CPU: tests/fake_hip.py): handles of different sizes, whose launches
may come in any order and from any thread, ask for the same."""
import numpy as np

from fake_hip import fake, fake_lib  # noqa: F401
from gpu_common import make_engine, synthetic_state


def test_handles_of_all_sizes_ask_for_the_same(fake):
    beyond = set()
    for nx, ny, depth in ((400, 300, 2), (330, 250, 2), (430, 320, 2), (900, 700, 1), (64, 48, 2)):
        st = synthetic_state(nx, ny, 5, ice_prob=0.7)
        z = np.zeros(st.na)
        with make_engine(st, 120) as eng:
            if depth == 1:
                eng.set_fused_depth(1)
                eng.set_tiling(62, 39, 512)
            fake.launches()
            eng.run(500)
            eng.adjoint_run(4, z, z)
            eng.tangent_run(4, z, z)
            beyond |= {n for n, _, _, lds in fake.launches() if lds > 64 * 1024}
    asked = {}
    for n, v in fake.attributes():
        asked.setdefault(n, set()).add(v)
    assert beyond and beyond <= set(asked)
    assert {n: v for n, v in asked.items() if len(v) > 1} == {}
