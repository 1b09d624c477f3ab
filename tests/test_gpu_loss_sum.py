"""The misfit is summed per workgroup on the device and over workgroups on the
host, in evp1d_loss, the gradient and the tangent: against the exactly rounded
sum of the same terms, at sizes around one workgroup and with an almost empty
last one.  Bound: each term passes at most 9 additions in double (6 within a
wavefront, 3 between them) before the host's long double, and the result is
rounded once: 10 units of 2^-53, and one for the terms of second order."""
import math

import numpy as np
import pytest

from gpu_common import fetch_state, make_engine, synthetic_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(1, 1), (17, 15), (16, 16), (257, 1), (400, 300)])
def test_loss_against_exact_sum(gpu, nx, ny):
    st = synthetic_state(nx, ny, seed=5, land_frac=0.0, ice_prob=1.0)
    r = np.random.default_rng(3)
    ut, vt = 0.1 * r.standard_normal(st.na), 0.1 * r.standard_normal(st.na)
    nsub = 4
    with make_engine(st, nsub) as eng:
        g = eng.adjoint_run(nsub, ut, vt)
        got = fetch_state(eng, st)
        values = [g["loss"], eng.loss(ut, vt)]
    with make_engine(st, nsub) as eng:
        values.append(eng.tangent_run(nsub, ut, vt)[0])
    at = np.asarray(st.skipU)[: st.na] == 0
    ex, ey = got.f["uvel"][: st.na] - ut, got.f["vvel"][: st.na] - vt
    want = math.fsum((0.5 * (ex * ex + ey * ey))[at])
    for v in values:
        assert abs(v - want) <= 11 * 2.0 ** -53 * want
