"""Split cohorts larger than the memory-side cache: groups of grids one after the other, bit for bit the whole."""
import numpy as np
import pytest

from torchfdtd_amd import workloads as W
from torchfdtd_amd.models import Monitor

SHAPES = [(24, 20, 16), (30, 18, 22), (20, 27, 18), (33, 24, 17), (18, 18, 30)]


def cohort(precision, traced=False):
    from torchfdtd_amd.batch import Cohort, Launch
    rng = np.random.default_rng(11)
    projects, designs = [], []
    for i, shape in enumerate(SHAPES):
        p = W.uneven_grid(shape, steps=41, pml=4+i % 2, frequencies=3+i, precision=precision, inset_cells=6, name=f'g{i}')
        if i == 1:
            p.monitors = []
        if i == 2 and precision == 'float32':
            p.monitors[0].dft_precision = 'field'
        if traced:
            p.monitors.append(Monitor(id='probe', center=(0, 0, 0), component='Ez'))
        projects.append(p)
        designs.append(W.design_epsilon(p, W.binary_design(rng, shape=(8, 8)), depth=4))
    return Cohort(projects, Launch('split'), epsilons=designs)


@pytest.mark.gpu
@pytest.mark.parametrize('precision', ['float32', 'float64'])
@pytest.mark.parametrize('share', [2, 3, 100])
def test_grouped_blocks_equal_whole_steps(gpu, monkeypatch, precision, share):
    """Graphs of a width and a remainder, and eager blocks; a group per grid, a few, and none that a grid fits."""
    from torchfdtd_amd import batch
    whole = cohort(precision)
    assert whole.groups == []
    for _ in range(41):
        whole.step()
    total = sum(t.numel()*t.element_size() for g in whole.grids for t in (g.E, g.H, g.inverse_permittivity, *g.psi_buffers.values()))
    monkeypatch.setattr(batch, 'WHOLE_BYTES', 0)
    monkeypatch.setattr(batch, 'GROUP_BYTES', max(1, total//share))
    replayed, eager = cohort(precision), cohort(precision)
    assert sum(grids for _, grids, _ in replayed.groups) == len(SHAPES) and 2 <= len(replayed.groups) <= len(SHAPES)
    graphs = replayed.graphs(8)
    graphs.advance(41)
    eager.advance(13)
    eager.advance(28)
    assert int(replayed.counter) == int(eager.counter) == 41
    assert replayed.digest() == whole.digest() and eager.digest() == whole.digest()


@pytest.mark.gpu
def test_cohorts_with_traces_stay_whole(gpu, monkeypatch):
    from torchfdtd_amd import batch
    whole = cohort('float32', True)
    whole.advance(41)
    monkeypatch.setattr(batch, 'WHOLE_BYTES', 0)
    monkeypatch.setattr(batch, 'GROUP_BYTES', 1)
    other = cohort('float32', True)
    assert other.groups == []
    other.graphs(8).advance(41)
    assert other.digest() == whole.digest()
