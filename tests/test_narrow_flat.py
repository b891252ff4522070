"""Flat grids narrower than a patch: which of them the patches take (host rule, CPU)."""
import ctypes

import pytest

from torchfdtd_amd import _native as N


def takes(nx, ny, dtype=N.F32):
    """Whether tfdtd_flat_steps takes a grid of one z plane (it only asks: nothing is launched)."""
    lib = N.load_library()
    e, h = N.HalfStep(), N.HalfStep()
    for d, family in ((e, N.FAMILY_E), (h, N.FAMILY_H)):
        d.dtype, d.family, d.nx, d.ny, d.nz, d.inverse_stride = dtype, family, nx, ny, 1, int(family == N.FAMILY_E)
        d.src, d.dst, d.inverse = (16, 32, 48) if family == N.FAMILY_E else (32, 16, 64)
    observe = N.Observe()
    observe.dtype, observe.counter = dtype, 80
    status = lib.tfdtd_flat_steps(ctypes.byref(e), ctypes.byref(h), ctypes.byref(observe), None, None, None, 0, None)
    assert status in (0, N.EUNSUPPORTED), N.last_error()
    return status == 0


@pytest.mark.parametrize('dtype', [N.F32, N.F64])
def test_long_grids_narrower_than_a_patch_keep_half_steps(dtype):
    for narrow, long in ((5, 60000), (8, 60000), (5, 1000000), (9, 1000000)):
        assert not takes(narrow, long, dtype) and not takes(long, narrow, dtype)
    for narrow, long in ((5, 40), (5, 40000), (8, 40000), (12, 100000), (12, 1000000), (24, 1000000), (160, 120), (3000, 3000)):
        assert takes(narrow, long, dtype) and takes(long, narrow, dtype)
