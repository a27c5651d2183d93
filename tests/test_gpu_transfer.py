"""Host arrays up and down through the pinned buffers.

Sizes: the smallest grid, rows shorter and longer than a wavefront and than a
block's 256 columns, one run, two runs, and transfers above four buffers,
which several threads share (16 MB; here 24 and 137 MB with ragged last runs).
Every value comes back as it went up, and only where it belongs: the planes
not written keep theirs.
"""
import ctypes

import numpy as np
import pytest

import cueva

pytestmark = pytest.mark.gpu

GRIDS = [(8, 8), (9, 300), (51, 20), (243, 17), (244, 64), (600, 31), (333, 640), (509, 1021)]


@pytest.mark.parametrize("ni,nj", GRIDS, ids=["%dx%d" % g for g in GRIDS])
def test_planes_come_back_as_they_went_up(ni, nj):
    print("transfer", ni, nj, flush=True)
    p = cueva.kh_params(ni, nj)
    rng = np.random.default_rng(ni * 1000 + nj)
    shape = (p.jmax + 13, p.imax + 13)
    a = rng.normal(size=(14,) + shape)
    c = rng.normal(size=(5,) + shape)
    inner = np.s_[:, 6:6 + nj + 1, 6:6 + ni + 1]
    with cueva.Solver(p) as s:
        s.upload_cons(c)
        s.upload(a)
        pr, co = s.download()
        assert np.array_equal(pr[inner], a[inner])
        assert np.array_equal(co, c)
        assert np.array_equal(s.download(cons=False), pr)
        for k in (0, 7, 13):
            assert np.array_equal(s.plane(0, k), pr[k])
        assert np.array_equal(s.plane(1, 4), c[4])
        assert not s.plane(1, 5).any()  # W: neither upload touches it
        # a second state over the first, from another array
        s.upload(-a)
        assert np.array_equal(s.download(cons=False)[inner], -a[inner])
        assert np.array_equal(s.plane(1, 0), c[0])


def test_device_memory_in_place_of_a_host_array():
    p = cueva.kh_params(40, 30)
    a = np.random.default_rng(5).normal(size=(14, p.jmax + 13, p.imax + 13))
    rt = ctypes.CDLL("libamdhip64.so.7")
    with cueva.Solver(p) as s:
        d = ctypes.c_void_p()
        assert rt.hipMalloc(ctypes.byref(d), ctypes.c_size_t(a.nbytes)) == 0
        assert rt.hipMemcpy(d, a.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(a.nbytes), 1) == 0
        ptr = ctypes.cast(d, ctypes.POINTER(ctypes.c_double))
        assert s.lib.cueva_upload_prims(s.ctx, ptr) == 0
        got = s.download(cons=False)
        rt.hipFree(d)
    inner = np.s_[:, 6:6 + p.jmax + 1, 6:6 + p.imax + 1]
    assert np.array_equal(got[inner], a[inner])
