"""Grids whose (y, z) planes leave the march's wavefronts mostly idle keep the general half step.

Which step a grid took shows in the stepper's shadow counter (only the marched E launch writes it), and in the
workgroups of a packed batch (512 cells each for the general step).
"""
import ctypes

import pytest
import torch

from torchfdtd_amd import _native as N


def packed(shapes, dtype=N.F32):
    lib, count = N.load_library(), len(shapes)
    steps = (N.HalfStep*count)()
    for d, (nx, ny, nz) in zip(steps, shapes):
        d.dtype, d.family, d.nx, d.ny, d.nz, d.inverse_stride = dtype, N.FAMILY_E, nx, ny, nz, 1
        d.src = d.dst = d.inverse = 16
    nbytes = lib.tfdtd_batch_table_bytes(count, dtype)
    prefix = (ctypes.c_int32*(count+1))()
    N.check(lib.tfdtd_batch_pack(steps, count, (ctypes.c_ubyte*nbytes)(), nbytes, prefix), 'pack')
    return [prefix[k+1]-prefix[k] for k in range(count)]


def test_a_batch_of_thin_grids_takes_the_general_step():
    strip, full = (2000, 5, 1), (40, 64, 32)
    assert packed([strip]*4) == [500]*4                    # 472,000 idle lanes: a wavefront per plane
    assert packed([strip]*5) == [20]*5
    assert packed([strip]*5+[full]) == [20]*5+[320]        # planes that fill their lanes march beside them
    assert packed([(100, 10, 10)]*187) == [50]*187 and packed([(100, 10, 10)]*188) == [20]*188
    assert packed([(100, 11, 10)]*400) == [50]*400         # 110 of 128 lanes
    assert packed([(100, 10, 10)]*400, N.F64) == [50]*400 and packed([(100, 17, 5)]*400, N.F64) == [17]*400


@pytest.mark.gpu
@pytest.mark.parametrize('shape,precision,faces,marches', [
    ((4000, 5, 1), 'float32', {'y': 'periodic'}, True), ((40000, 5, 1), 'float32', {'y': 'periodic'}, False),
    ((60000, 5, 5), 'float32', {'y': 'periodic', 'z': 'periodic'}, False), ((40000, 32, 1), 'float32', {}, True),
    ((60000, 5, 5), 'float64', {'y': 'periodic', 'z': 'periodic'}, True), ((60000, 16, 1), 'float64', {}, False),
    ((2732, 2048, 1), 'float64', {}, False), ((2730, 2048, 1), 'float64', {}, True), ((2732, 2048, 1), 'float32', {}, True)])
def test_which_step_a_grid_takes(gpu, shape, precision, faces, marches):
    from test_plane_march import separate_coefficients, state, stepper
    run, general = (stepper(shape, precision, 'cell', faces, 2) for _ in range(2))
    kept = separate_coefficients(general)
    for _ in range(3):
        run.step()
        general.step()
    torch.cuda.synchronize()
    assert kept and int(general.shadow) == 0 and int(general.counter) == int(run.counter) == 3
    assert int(run.shadow) == (2 if marches else 0)
    for a, b in zip(state(run), state(general)):
        assert torch.equal(a, b)
