"""A context that has held NaN gives a new state the values a fresh one gives.

``cueva_upload_prims`` starts a context again, so nothing of the state before
may reach the steps after it.  MIRK2's closing electric field multiplies the
last stage's B by that stage's velocity, which is zero without REC_PRIM = 1:
finite values left there by an earlier state do no harm, NaN does.  One stage
(order 1) is the case where the last stage is also the first, whose planes the
mixed marching step need not keep; two stages and MIRK1 stand beside it.
"""
import numpy as np
import pytest

import cueva

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [cueva.FP64, cueva.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("order,mirk", [(1, 1), (1, 2), (2, 2)])
def test_new_state_after_nan(order, mirk, precision):
    p, prims = cueva.kh_problem(40, 60, sigma=10.0, flux_solver=cueva.HLL, order=order, mirk=mirk, precision=precision)
    p.cfl = 0.1
    print("reuse after NaN", order, mirk, precision, flush=True)
    bad = prims.copy()
    bad[2:5, 20:40, 15:30] = np.nan
    with cueva.Solver(p) as s:
        s.upload(prims)
        s.step(2)
        want = s.download()
    assert all(np.isfinite(a).all() for a in want)
    with cueva.Solver(p) as s:
        s.upload(bad)
        s.step_status(1)  # with or without a stop: the stage state that stays holds NaN
        assert np.isnan(s.plane(2, 2)).any()
        s.upload(prims)
        s.step(2)
        got = s.download()
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
