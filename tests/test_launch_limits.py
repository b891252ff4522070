"""Calls at the limit of a launch, fewer than 2^32 threads, take the path that still fits it (host rules, CPU)."""
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
