"""Blocked plane accumulation against accumulation every step: frequencies that do not fill a group of four,
downsampled windows and blocks left unfinished."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('frequencies,downsample,steps', [(1, 1, 33), (4, 3, 40), (5, 1, 31), (13, 2, 65)])
def test_blocked_sums_equal_step_by_step_sums(gpu, frequencies, downsample, steps):
    from torchfdtd_amd import FieldMonitor, Project, Region, Source, SpectrumSettings
    from torchfdtd_amd.solver import Stepper
    region = Region(dimension='3d', size=(1.7, 1.5, 1.6), mesh=.1, pml_cells=3, steps=70, backend='cuda')
    spectrum = SpectrumSettings(sampling='wavelength', frequency_points=frequencies, wavelength_start=1, wavelength_stop=2, apodization='none')
    monitor = FieldMonitor(id='m', center=(.2, 0, 0), normal='x', size=(0, .7, .8), dft_precision='float64', spectrum=spectrum,
                           time_downsample=downsample)
    project = Project(region=region, sources=[Source(id='s', wavelength=1, pulse_cycles=1)], monitors=[monitor])
    values = []
    for block in (32, 1):
        run = Stepper(project)
        run.planes[0].block = block
        run._describe()
        for _ in range(steps):
            run.step()
        run.planes[0].flush()
        values.append(run.planes[0].value.clone())
    torch.cuda.synchronize()
    # The same FP64 products, summed in another order: 1e-12 of the largest entry, as the oracle comparisons.
    scale = float(values[1].abs().max())
    assert scale > 0
    assert float((values[0]-values[1]).abs().max()) <= 1e-12*scale
