"""The curl record made by the E launch against a launch of its own before the step, bit for bit."""
import ctypes

import pytest
import torch

from test_plane_march import separate_coefficients, state, stepper

pytestmark = pytest.mark.gpu

# The whole grid, boxes of one cell, in a corner's slabs and across the 64-cell columns; one and three permittivity
# values, odd and even x, periodic edges, flat grids.
CASES = [((17, 12, 16), 'float32', 'cell', {}, None), ((66, 65, 63), 'float32', 'yee', {}, ((0, 1), (64, 65), (62, 63))),
         ((13, 11, 17), 'float64', 'cell', {'y': 'periodic'}, ((1, 12), (0, 5), (3, 17))),
         ((71, 61, 67), 'float64', 'yee', {'x': 'periodic'}, ((30, 71), (0, 61), (10, 43))),
         ((65, 66, 64), 'float32', 'cell', {'z': 'periodic', 'x': 'pec'}, ((0, 65), (1, 65), (0, 64))),
         ((40, 129, 1), 'float32', 'cell', {}, ((3, 38), (0, 100), (0, 1)))]


@pytest.mark.parametrize('separate', [False, True])
@pytest.mark.parametrize('shape,precision,sampling,faces,box', CASES)
def test_recorded_step_equals_the_separate_record(gpu, shape, precision, sampling, faces, box, separate):
    from torchfdtd_amd import _native as N
    from torchfdtd_amd.grid import march_family
    from torchfdtd_amd.planning import periodic_axes
    box = box or tuple((0, n) for n in shape)
    runs = [stepper(shape, precision, sampling, faces, 13) for _ in range(2)]
    kept = separate_coefficients(runs[0]) if separate else None     # the general step: the record keeps its launch
    cells = [b-a for a, b in box]
    records = []
    for run in runs:
        g = run.grid
        out = torch.full((3, cells[0]*cells[1]*cells[2], 3), float('nan'), device=g.device, dtype=g.dtype)
        d = N.CurlRecord()
        d.e = march_family(g, False, g.psi_buffers[False], g.psi_buffers[False])
        d.dtype = N.F64 if g.dtype == torch.float64 else N.F32
        d.nx, d.ny, d.nz = shape
        d.H, d.record, d.modulus, d.counter = g.H.data_ptr(), out.data_ptr(), 3, run.counter.data_ptr()
        d.periodic_mask = sum(1 << a for a in periodic_axes(g.region))
        for a in range(3):
            d.box_lo[a], d.box_hi[a] = box[a]
        records.append((d, out))
    for _ in range(5):
        runs[0].step(records[0][0])
        N.check(runs[1].lib.tfdtd_record_curl(ctypes.byref(records[1][0]), N.stream_handle()), 'record')
        runs[1].step()
    torch.cuda.synchronize()
    assert kept is None or kept
    assert bool(torch.isfinite(records[0][1]).all()) and torch.equal(records[0][1], records[1][1])
    for a, b in zip(state(runs[0]), state(runs[1])):
        assert torch.equal(a, b)
