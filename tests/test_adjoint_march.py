"""The marched transposes and record against the NumPy oracle on grids past one plane a march.

Columns of the (y, z) plane with spare lanes, odd and even x under marches of two planes (4,096 column-planes and
more) and of one, each kind of edge, flat grids, and boxes off the grid's corner.
"""
import numpy as np
import pytest

from tests.test_adjoint import engine_gradient, oracle_gradient
from torchfdtd_amd.adjoint import AdjointOptions
from torchfdtd_amd.models import Boundaries, BoundaryFace, Monitor, Project, Region, Source

pytestmark = pytest.mark.gpu


def project_for(shape, precision, faces, steps):
    pairs = {axis+side: BoundaryFace(kind=kind) for axis, kind in faces.items() for side in ('_min', '_max')}
    region = Region(dimension='2d' if shape[2] == 1 else '3d', size=tuple(.1*n for n in shape), mesh=.1, pml_cells=3, precision=precision,
                    steps=steps, boundaries=Boundaries(**pairs), backend='cuda')
    return Project(region=region, sources=[Source(id='s', component='Ez', pulse_length=3e-15, pulse_offset=6e-15, time_definition='standard')],
                   monitors=[Monitor(id='a', center=(.1, .1, 0), component='Ez'), Monitor(id='b', center=(0, -.1, 0), component='Hy'),
                             Monitor(id='c', center=(-.1, 0, 0), component='Ex')])


@pytest.mark.parametrize('shape,precision,faces,per_component', [
    ((65, 65, 64), 'float64', {}, False), ((66, 64, 65), 'float32', {'z': 'pec'}, False), ((67, 63, 65), 'float64', {'x': 'periodic', 'y': 'periodic'}, True),
    ((13, 11, 17), 'float64', {'y': 'pec'}, True), ((15, 23, 1), 'float64', {}, False), ((131, 2050, 1), 'float64', {'x': 'periodic'}, False)])
def test_gradient_of_marched_grids_matches_the_oracle(gpu, shape, precision, faces, per_component):
    steps = 10
    project = project_for(shape, precision, faces, steps)
    rng = np.random.default_rng(5)
    eps = rng.uniform(1, 3, shape+((3,) if per_component else ())).astype(np.float64 if precision == 'float64' else np.float32)
    weights = rng.normal(size=(steps, 3))
    _, want, _ = oracle_gradient(project, eps, weights)
    _, got, _ = engine_gradient(project, eps, weights)
    tol = 1e-9 if precision == 'float64' else 2e-4       # of the largest entry, as tests/test_adjoint.py
    scale = np.abs(want).max()
    assert scale > 0
    np.testing.assert_allclose(got, want, rtol=0, atol=tol*scale)
    box = tuple((n//2-1, n//2+3) if n > 1 else (0, 1) for n in shape)
    _, part, _ = engine_gradient(project, eps, weights, AdjointOptions(design_box=box))
    inside = tuple(slice(a, b) for a, b in box)
    assert np.array_equal(part[inside], got[inside])


def test_plane_observers_are_numbered_as_they_first_appear(gpu):
    from torchfdtd_amd.adjoint import COMPONENTS, DifferentiablePlaneSimulation
    from torchfdtd_amd.models import FieldMonitor, SpectrumSettings
    from torchfdtd_amd.monitors import interpolation_map
    spectrum = SpectrumSettings(sampling='wavelength', frequency_points=2, wavelength_start=1, wavelength_stop=2, apodization='none')
    planes = [('x', (.2, 0, 0), (0, .8, .8)), ('x', (.23, .1, 0), (0, .5, .6)), ('y', (0, .1, 0), (.7, 0, .6))]
    project = Project(region=Region(dimension='3d', size=(1.7, 1.6, 1.9), mesh=.1, pml_cells=3, steps=20), sources=[Source(id='s')],
                      monitors=[FieldMonitor(id=f'm{i}', normal=n, center=c, size=s, spectrum=spectrum) for i, (n, c, s) in enumerate(planes)])
    model = DifferentiablePlaneSimulation(project)
    expected = []
    for _, _, plan, maps in model.plans:
        for component, (numbers, _) in zip(COMPONENTS, maps):
            indices, _ = interpolation_map(project.region, component, plan['points_um'])
            for flat, number in zip(indices.reshape(-1).tolist(), numbers.reshape(-1).tolist()):
                if number == len(expected):
                    expected.append((component[0] == 'H', flat))
                assert expected[number] == (component[0] == 'H', flat)
    assert model.observers == expected and len(set(expected)) == len(expected)
    assert model.components == tuple('H' if m else 'E' for m, _ in expected)
