"""The stage planes that cueva_download_plane returns after cueva_step.

Inside the marching step a stage state is kept only as far as its launches
read it (J_z and, in the mixed form, D tau S J and the first stage's psi phi
B q in FP64 are left out); the state that stays after a call, and that of a
failing launch, are kept or formed again in full.  Every plane is compared
with the face-plane path (CUEVA_MARCH=0), which keeps all of them: interior
points for calls of one and of several steps, schemes of one to four stages,
with and without the primitive reconstruction at the start of a step, solvers
with filled and with zero J ghosts; and at a failure in either stage.
"""
import os

import numpy as np
import pytest

import crafted
import cueva

pytestmark = pytest.mark.gpu

STAGE = [k for k in range(20) if not 5 <= k <= 7]  # EXA..EZA are not part of it
CASES = {
    "hllc": dict(flux_solver=cueva.HLLC),
    "hlle_bz": dict(flux_solver=cueva.HLLE, rec_mp=1, bz0=0.1),
    "lax_primrec": dict(flux_solver=cueva.LAX, sigma=1.0e3, primitive_rec=1),
    "hllc_mc": dict(flux_solver=cueva.HLLC_MCL, sigma=1.0e3),
    "hll_mirk1": dict(flux_solver=cueva.HLL, sigma=1.0e3, order=1, mirk=1),
    "hll_ssp3": dict(flux_solver=cueva.HLL, sigma=1.0e3, order=4),
}


def planes(p, prims, steps, march, expect=0):
    old = os.environ.get("CUEVA_MARCH")
    os.environ["CUEVA_MARCH"] = "1" if march else "0"
    try:
        with cueva.Solver(p) as s:
            s.upload(prims)
            rc = s.step_status(steps)
            where = s.last_error()[1]
            st = np.stack([s.plane(2, k) for k in STAGE])
            pr = s.download(cons=False)
    finally:
        if old is None:
            del os.environ["CUEVA_MARCH"]
        else:
            os.environ["CUEVA_MARCH"] = old
    assert (rc != 0) == bool(expect), rc
    sl = np.s_[:, 6:6 + p.jmax + 1, 6:6 + p.imax + 1]
    return rc, where, st[sl], pr[sl]


@pytest.mark.parametrize("steps", [1, 2, 3])
@pytest.mark.parametrize("precision", [cueva.FP64, cueva.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_stage_planes_after_a_call(name, precision, steps):
    kw = dict(CASES[name])
    sigma = kw.pop("sigma", 1.0e6)
    p, prims = cueva.kh_problem(70, 130, sigma=sigma, precision=precision, **kw)
    print("stage planes", name, precision, steps, flush=True)
    _, _, a, pa = planes(p, prims, steps, True)
    _, _, b, pb = planes(p, prims, steps, False)
    assert np.array_equal(pa, pb)
    bad = [STAGE[k] for k in range(len(STAGE)) if not np.array_equal(a[k], b[k])]
    assert not bad


@pytest.mark.parametrize("precision", [cueva.FP64, cueva.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("fs", [cueva.HLL, cueva.HLLC], ids=["recovery", "faces"])
def test_stage_planes_at_a_failure(fs, precision):
    """Data whose recovery (HLL) or face solve (HLLC) stops the first of two steps."""
    p, prims = cueva.kh_problem(32, 64, sigma=1.0e3, flux_solver=fs, rotated=True, precision=precision)
    crafted.spin(prims)
    print("stage planes at a failure", fs, precision, flush=True)
    ra, wa, a, pa = planes(p, prims, 2, True, expect=1)
    rb, wb, b, pb = planes(p, prims, 2, False, expect=1)
    assert (ra, wa) == (rb, wb) and wa[0] == 1
    bad = [STAGE[k] for k in range(len(STAGE)) if not np.array_equal(a[k], b[k], equal_nan=True)]
    assert not bad
