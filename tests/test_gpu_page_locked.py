"""Read-back into page-locked memory (written by the gather itself) against
read-back into ordinary memory (a copy), bit for bit: the 1D list, members of
a batch and the 2D path, at the start of an allocation, up to its last value,
and at an odd address, which takes the copy."""
import ctypes

import numpy as np
import pytest

import evp1d
from evp1d import synth
from gpu_common import make_engine, synthetic_state
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DP = ctypes.POINTER(ctypes.c_double)


def _check(lib, get, want):
    """get(pointer, n) writes n values; want: the same from ordinary memory."""
    n, pad = want.size, 64
    ptr = ctypes.c_void_p()
    assert lib.evp1d_host_alloc(8 * (n + pad), ctypes.byref(ptr)) == 0
    try:
        raw = np.frombuffer((ctypes.c_char * (8 * (n + pad))).from_address(ptr.value), np.uint8)
        for byte in (0, 8 * pad, 12):
            raw[:] = 0xab
            assert get(ctypes.cast(ptr.value + byte, DP), n) == 0
            assert (raw[byte:byte + 8 * n] == want.view(np.uint8)).all(), f"at byte {byte}"
            assert (raw[:byte] == 0xab).all() and (raw[byte + 8 * n:] == 0xab).all()
        del raw
    finally:
        assert lib.evp1d_host_free(ptr) == 0


@pytest.mark.parametrize("nx,ny", [(1, 1), (23, 17), (300, 211)])
def test_list_and_member(gpu, nx, ny):
    st = synthetic_state(nx, ny, seed=4, land_frac=0.1 if nx > 1 else 0.0)
    with make_engine(st, 4) as eng:
        eng.run(4)
        for f in ("uvel", "vvel", "stressp_1", "str8", "Tbu"):
            _check(eng.L, lambda p, n: eng.L.evp1d_get_field(eng.h, evp1d.FIELD_ID[f], p, n), eng.get_field(f))
            _check(eng.L, lambda p, n: eng.L.evp1d_get_field_member(eng.h, 0, evp1d.FIELD_ID[f], p, n),
                   eng.get_field(f))


@pytest.mark.parametrize("nx,ny,nblocks", [(5, 4, 1), (90, 61, 3)])
def test_blocks(gpu, nx, ny, nblocks):
    st = O.pack_v0(synth.make_grid(nx, ny, 8, land_frac=0.1), nblocks)
    with evp1d.Engine2D(st.nxb, st.nyb, st.nblocks, evp1d.set_evp_parameters(120)) as eng:
        eng.load_state(st)
        eng.run(4)
        for f in ("uvel", "stressm_3", "str5"):
            _check(eng.L, lambda p, n: eng.L.evp2d_get_field(eng.h, evp1d.FIELD2D_ID[f], p, n),
                   np.asfortranarray(eng.get_field(f)).ravel(order="F"))
