"""The joint face evaluation (limiters of both sides, positivity fallback) on rough data.

The Kelvin-Helmholtz cases keep most wavefronts on the unlimited values and
never leave the positive range.  Here every field is random from point to
point, with jumps, extrema of all signs, equal neighbours, values near the
smallest positive number, negative densities and pressures, and (second
case) NaN and infinities, so that every limiter branch and the positivity
fallback run in lanes beside lanes that skip them.  The face fluxes are
compared bit for bit with the oracle's, which evaluates mp5.f95:79-216 as it
stands; where a flux is NaN, NaN is all that is compared.
"""
import sys

import numpy as np
import pytest

import cueva
from oracle.binding import Oracle

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rough(p, seed, special):
    rng = np.random.default_rng(seed)
    shape = (14, p.jmax + 13, p.imax + 13)
    a = rng.normal(scale=0.1, size=shape)
    a[rng.random(shape) < 0.2] = 0.05  # equal neighbours
    a[rng.random(shape) < 0.05] *= 1.0e-12
    a[:2][rng.random((2,) + shape[1:]) < 0.1] = 3.0e-308
    a[5:8] = rng.uniform(-0.3, 0.3, (3,) + shape[1:])
    a[12:] = np.exp(rng.normal(scale=1.5, size=(2,) + shape[1:]))  # far from the smooth range
    calm = np.s_[:, : shape[2] // 3]
    for k in (12, 13):
        a[k][calm] = 1.0 + 0.01 * rng.normal(size=a[k][calm].shape)
        a[k][rng.random(shape[1:]) < 0.01] *= -1.0
    if special:
        for v in (np.nan, np.inf, -np.inf):
            a[rng.random(shape) < 4.0e-4] = v
    return a


@pytest.mark.parametrize("special", [False, True], ids=["finite", "nan_inf"])
@pytest.mark.parametrize("rec", [0, 1, 2], ids=["mp5", "mp7", "mp9"])
def test_face_fluxes_of_rough_data(rec, special):
    # order 1 with MIRK1 has one stage: its fluxes are those of the uploaded state
    p = cueva.kh_params(70, 45, sigma=1.0e3, flux_solver=cueva.HLL, rec_mp=rec, order=1, mirk=1)
    prims = rough(p, 3 + rec, special)
    say("rough data, MP", 5 + 2 * rec, "special" if special else "finite")
    L = cueva.load()
    with cueva.Solver(p) as s:
        x = s.ctx
        s.upload(prims)
        for call in (lambda: L.cueva_boundary(x, cueva.abi.BND_PRIM, 1), lambda: L.cueva_startconvar(x),
                     lambda: L.cueva_cleanvarint(x), lambda: L.cueva_swap1(x), lambda: L.cueva_varint(x, 1),
                     lambda: L.cueva_electricvarint(x, 1), lambda: L.cueva_flowinit(x, 1), lambda: L.cueva_flux(x, 1)):
            assert call() == 0
        got = np.stack([s.plane(3 + q // 14, q % 14) for q in range(28)])
    o = Oracle(p)
    o.upload(prims)
    o.step_status(1)  # its recovery may stop on such data; the face pass came before
    want = np.stack([o.face(q // 14, q % 14) for q in range(28)])
    sl = np.s_[:, 5:5 + p.jmax + 2, 5:5 + p.imax + 2]
    got, want = got[sl], want[sl]
    bad = [q for q in range(28) if not np.array_equal(got[q], want[q], equal_nan=True)]
    say("NaN share", float(np.isnan(want).mean()), "differing slots", bad)
    assert special == bool(np.isnan(want).any())
    assert not bad
