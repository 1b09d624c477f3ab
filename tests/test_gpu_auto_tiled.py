"""AUTO's own tiles against the reference's output files and the oracle.  A
first short run takes no tiles, so they are planned before it here; that it
then takes them, which no result shows, is what test_auto_form.py holds."""
import json

import numpy as np
import pytest

from evp1d import synth
from gpu_common import (GOLD, assert_state_bitexact, fetch_state, golden_cases, load_golden, make_engine,
                        oracle_params, synthetic_state)
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _run_planned(st, ndte):
    with make_engine(st, ndte) as eng:
        assert eng.get_fused_depth()["active"]   # plans the tiles
        eng.run(ndte)
        return fetch_state(eng, st)


@pytest.mark.parametrize("case", golden_cases())
def test_golden_outputs(gpu, case):
    st, ndte, want_stress, want_stepu = load_golden(case)
    assert O.output_bytes(_run_planned(st, ndte)) == (want_stress, want_stepu)


def test_evp_c0_md5(gpu):
    rec = json.loads((GOLD / "golden.json").read_text())["evp_c0"]
    w = synth.WORKLOADS["evp_c0"]
    a, b = O.output_bytes(_run_planned(synthetic_state(w["nx"], w["ny"], w["seed"]), w["ndte"]))
    assert (O.md5(a), O.md5(b)) == (rec["output_stress_md5"], rec["output_stepu_md5"])


def test_new_flags_with_a_copy_list(gpu):
    st = synthetic_state(70, 52, seed=57)
    r = np.random.default_rng(19)
    ghosts = np.arange(st.na + 1, st.navel + 1, dtype=np.int32)
    dst = r.choice(ghosts, size=ghosts.size // 2, replace=False).astype(np.int32)
    src = r.integers(0, st.na + 1, size=dst.size).astype(np.int32)
    lib, p = oracle_params(st, 9)
    want = st.copy()
    with make_engine(st, 9) as eng:
        eng.set_halo(dst, src)
        for nsub in (9, 7, 8):
            want.skipT[:] = st.skipT | (r.random(st.na) < 0.3)
            want.skipU[:] = st.skipU | (r.random(st.na) < 0.2)
            eng.set_skip("skipT", want.skipT)
            eng.set_skip("skipU", want.skipU)
            assert eng.get_fused_depth()["active"]   # plans the tiles for them
            eng.run(nsub)
            lib.run(p, want, nsub, halo=(dst, src))
            assert_state_bitexact(fetch_state(eng, st), want)
