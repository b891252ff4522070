"""Calls at the limit of a launch, fewer than 2^32 threads, take the path that still fits it (host rules, CPU)."""
import ctypes

import pytest

from torchfdtd_amd import _native as N


def test_a_march_beyond_one_launch_is_left_to_the_general_step():
    from test_thin_planes import packed
    # One wavefront per 64-cell column and two planes; the general step takes 512 cells a workgroup.
    inside, beyond = (1 << 27)-16, (1 << 27)+2
    assert packed([(inside, 60, 1)]) == [inside//8]
    assert packed([(beyond, 60, 1)]) == [-(-beyond*60//512)]


def test_patches_beyond_one_launch_are_left_to_half_steps():
    from test_narrow_flat import takes
    for dtype in (N.F32, N.F64):
        assert takes(49000, 49000, dtype) and not takes(50000, 50000, dtype)


@pytest.mark.parametrize('rows', [(1 << 31)-1, (1 << 31)-256])
def test_rows_within_a_workgroup_of_the_last_count_are_left_to_the_general_kernel(rows):
    """Refused before any launch, as the sizes of the last workgroup's rows do not fit 32 bits."""
    from torchfdtd_amd.surrogate import ConvShape
    lib = N.load_library()
    narrow = ConvShape(rows, 1, 1, 1, 1, 1, 1, 1, 0, 32)
    x, weight, out = 1 << 20, 1 << 21, 1 << 22
    assert lib.tfdtd_conv_forward_rows(ctypes.byref(narrow), x, N.CONV_BF16, weight, None, None, 0, out, None, None, None) == N.EUNSUPPORTED
    wide = ConvShape(rows, 1, 1, 1, 8, 8, 1, 1, 0, 32)
    assert lib.tfdtd_conv_dgrad_rows(ctypes.byref(wide), x, weight, None, out, None) == N.EUNSUPPORTED
