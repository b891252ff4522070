"""The plane march of the half steps against the general half step, bit for bit.

A descriptor whose two terms of an axis share one coefficient block takes the plane march; giving one
term a copy of its coefficients (the same values elsewhere) sends the same step down the general path.
Both round every operation in the same order, so fields and CPML memory must be equal.
"""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def project_for(shape, precision, sampling, faces):
    from torchfdtd_amd import Boundaries, BoundaryFace, Project, Region, Source
    pairs = {axis+side: BoundaryFace(kind=kind) for axis, kind in faces.items() for side in ('_min', '_max')}
    region = Region(dimension='2d' if shape[2] == 1 else '3d', size=tuple(.1*n for n in shape), mesh=.1, pml_cells=3, steps=20,
                    precision=precision, material_sampling=sampling, boundaries=Boundaries(**pairs), backend='cuda')
    return Project(region=region, sources=[Source(id='e', component='Ez'), Source(id='h', component='Hy', center=(.1, .1, 0)),
                                           Source(id='sheet', kind='plane', normal='x', center=(-.2, 0, 0), size=(0, .3, .3), component='Ey')])


def stepper(shape, precision, sampling, faces, seed):
    from torchfdtd_amd.solver import Stepper
    rng = np.random.default_rng(seed)
    samples = (3,) if sampling == 'yee' else ()
    run = Stepper(project_for(shape, precision, sampling, faces), epsilon=rng.uniform(1, 4, (*shape, *samples)), one_pass=False)
    gen = torch.Generator(device='cuda').manual_seed(seed)
    for t in (run.grid.E, run.grid.H, *run.grid.psi_buffers.values()):
        t.copy_(torch.randn(t.shape, generator=gen, device='cuda', dtype=t.dtype))
    return run


def separate_coefficients(run):
    """The run's descriptors with every other segment's coefficients in copies of their own."""
    kept = []
    for step in (run.e_step, run.h_step):
        forward = step is run.h_step
        entries = [e for key, group in run.grid.cpml.items() if key[0] == forward for e in group]
        by_psi = {e['psi'].data_ptr(): e for e in entries}
        for k in range(0, step.nseg):
            entry = by_psi[step.seg[k].psi]
            copies = [entry[n].clone() for n in ('b', 'c', 'inv_k')]
            kept.append(copies)
            step.seg[k].b, step.seg[k].c, step.seg[k].inv_k = (c.data_ptr() for c in copies)
    return kept


def state(run):
    return [run.grid.E, run.grid.H, *run.grid.psi_buffers.values()]


# Planes of one cell less and more than whole 64-cell columns, odd and even x under both march lengths,
# one and three permittivity values per cell, each kind of edge, and flat grids.
CASES = [((17, 12, 16), 'float32', 'cell', {}), ((66, 65, 63), 'float32', 'cell', {}), ((67, 64, 64), 'float32', 'yee', {}),
         ((13, 11, 17), 'float64', 'cell', {'y': 'periodic'}), ((71, 61, 67), 'float64', 'yee', {'x': 'periodic', 'y': 'periodic'}),
         ((70, 63, 65), 'float32', 'cell', {'z': 'pec', 'y': 'pec'}), ((65, 66, 64), 'float32', 'cell', {'x': 'pec', 'z': 'periodic'}),
         ((11, 11, 1), 'float32', 'cell', {}), ((161, 1999, 1), 'float32', 'cell', {'x': 'periodic'}),
         ((129, 2112, 1), 'float64', 'yee', {'y': 'pec'})]


@pytest.mark.parametrize('shape,precision,sampling,faces', CASES)
def test_march_equals_the_general_step(gpu, shape, precision, sampling, faces):
    march, general = (stepper(shape, precision, sampling, faces, 7) for _ in range(2))
    kept = separate_coefficients(general)
    assert kept
    for _ in range(4):
        march.step()
        general.step()
    torch.cuda.synchronize()
    for a, b in zip(state(march), state(general)):
        assert torch.equal(a, b)


def test_batched_march_and_general_grids_together(gpu):
    from torchfdtd_amd import _native as N
    from torchfdtd_amd.solver import pack_table
    cases = [CASES[1], CASES[0], CASES[5]]
    runs, singles = ([stepper(*c, 11+i) for i, c in enumerate(cases)] for _ in range(2))
    kept = separate_coefficients(runs[1])
    lib = N.library()
    tables = [pack_table(lambda n: lib.tfdtd_batch_table_bytes(n, N.F32), lib.tfdtd_batch_pack,
                         [getattr(r, name) for r in runs], 1, gpu) for name in ('e_step', 'h_step')]
    for family, (table, prefix, host) in zip((N.FAMILY_E, N.FAMILY_H), tables):
        N.check(lib.tfdtd_batch_half_step(table.data_ptr(), prefix.data_ptr(), len(runs), int(host[0, -1]), N.F32, family,
                                          N.stream_handle()), 'batch')
        for run in singles:
            step = run.e_step if family == N.FAMILY_E else run.h_step
            N.check(lib.tfdtd_yee_half_step(ctypes.byref(step), N.stream_handle()), 'half step')
    torch.cuda.synchronize()
    assert kept
    for run, single in zip(runs, singles):
        for a, b in zip(state(run), state(single)):
            assert torch.equal(a, b)


@pytest.mark.parametrize('count', [1, 16, 17])
def test_observed_step_equals_the_separate_launches(gpu, count):
    """Traces folded into the H launch (up to 16) and read from the table beyond, against E, H, planes, traces and counter
    as separate launches: the same trace rows and counter, the last steps past the end of the rows."""
    from torchfdtd_amd import _native as N
    shape, lib = (13, 12, 17), N.library()
    runs = [stepper(shape, 'float32', 'cell', {}, 3) for _ in range(2)]
    last = 3*shape[0]*shape[1]*shape[2]-1
    flats = [0, last, 5, last-1, *np.random.default_rng(2).integers(0, last, 13).tolist()][:count]
    for run in runs:
        run.steps = 6
        run.set_trace_points([(k % 2 == 1, flat) for k, flat in enumerate(flats)])
    for _ in range(8):
        runs[0].step()
        N.check(lib.tfdtd_step_fused(ctypes.byref(runs[1].e_step), ctypes.byref(runs[1].h_step), runs[1].plane_table, 0,
                                     ctypes.byref(runs[1].observe), 1, N.stream_handle()), 'separate')
    torch.cuda.synchronize()
    assert runs[0].counter.item() == runs[1].counter.item() == 8
    assert torch.equal(runs[0].traces, runs[1].traces) and bool((runs[0].traces != 0).all())
    for a, b in zip(state(runs[0]), state(runs[1])):
        assert torch.equal(a, b)
