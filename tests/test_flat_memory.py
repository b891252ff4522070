"""The second buffer set of a flat run: made only where a block of steps runs, and done without where it does not fit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def project(interval):
    from test_plane_march import project_for
    p = project_for((40, 33, 1), 'float32', 'cell', {})
    p.region.steps, p.region.snapshot_interval = 60, interval
    return p


@pytest.mark.parametrize('width,interval,made', [(1, 20, False), (32, 20, False), (20, 20, True), (7, 20, True), (50, 60, True), (64, 60, False), (64, 30, False)])
def test_only_runs_that_replay_blocks_hold_a_second_set(gpu, monkeypatch, width, interval, made):
    from torchfdtd_amd import solver
    runs, init = [], solver.Stepper.__init__

    def spy(self, *args, **kwargs):
        init(self, *args, **kwargs)
        runs.append(self)
    monkeypatch.setattr(solver.Stepper, '__init__', spy)
    got = solver.Simulation(project(interval)).run(cuda_graph_steps=width)
    assert (runs[0].flat_set is not None) == made
    ref = solver.Simulation(project(interval)).run(cuda_graph=False)
    assert np.array_equal(got.electric, ref.electric) and np.array_equal(got.magnetic, ref.magnetic)


def test_a_state_that_fits_once_keeps_single_steps(gpu, monkeypatch):
    from torchfdtd_amd import solver
    ref = solver.Simulation(project(20)).run(cuda_graph_steps=20)
    flat, answers = solver.Stepper.flat, []

    def full(*args, **kwargs):
        raise torch.OutOfMemoryError('no memory for a second set')

    def without_room(self):
        with monkeypatch.context() as m:
            m.setattr(torch, 'empty_like', full)
            answers.append(flat(self))
        return answers[-1]
    monkeypatch.setattr(solver.Stepper, 'flat', without_room)
    got = solver.Simulation(project(20)).run(cuda_graph_steps=20)
    assert answers == [False]
    assert np.array_equal(got.electric, ref.electric) and np.array_equal(got.magnetic, ref.magnetic)


def test_the_report_counts_the_steps_of_blocks(gpu):
    from torchfdtd_amd.solver import Simulation
    steps = [Simulation(project(20)).run(cuda_graph_steps=width).summary['kernel_steps'] for width in (20, 7, 1)]
    # Barriers at 20, 40, 50 and 60.
    assert [s['flat'] for s in steps] == [40, 42, 0] and [s['split'] for s in steps] == [20, 18, 60]
    from test_plane_march import project_for
    cube = project_for((14, 13, 12), 'float32', 'cell', {})
    assert Simulation(cube).run(cuda_graph_steps=10).summary['kernel_steps'] == dict(two_step=0, one_pass=0, split=20, flat=0)
