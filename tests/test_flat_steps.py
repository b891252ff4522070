"""Several steps of a flat grid in one launch against single steps, bit for bit.

A patch of 32 x 32 cells takes 1 to 8 steps and owns its inner 30^2 to 16^2 cells: grids of one patch, of
whole patches and of one cell more, every kind of edge, step counts of every split into passes, and sizes
that take 8, 6 and 4 steps a pass.
"""
import pytest
import torch

from test_plane_march import state, stepper

pytestmark = pytest.mark.gpu

CASES = [((11, 11, 1), 'float32', 'cell', {}, (2, 3)), ((32, 16, 1), 'float32', 'yee', {}, (16, 50)),
         ((33, 17, 1), 'float64', 'cell', {}, (17, 9)), ((161, 119, 1), 'float32', 'cell', {}, (50, 2, 7)),
         ((31, 97, 1), 'float32', 'cell', {'x': 'periodic'}, (16, 33)), ((11, 7, 1), 'float64', 'yee', {'y': 'periodic'}, (16, 5)),
         ((5, 7, 1), 'float32', 'cell', {'x': 'periodic', 'y': 'periodic'}, (16, 15)),
         ((48, 65, 1), 'float32', 'cell', {'x': 'pec', 'y': 'pec'}, (16, 64)), ((65, 48, 1), 'float64', 'yee', {'y': 'pec'}, (31,)),
         ((401, 379, 1), 'float32', 'cell', {}, (25,)), ((1201, 1003, 1), 'float32', 'yee', {'x': 'periodic'}, (19,))]


@pytest.mark.parametrize('shape,precision,sampling,faces,counts', CASES)
def test_blocks_equal_single_steps(gpu, shape, precision, sampling, faces, counts):
    block, single = (stepper(shape, precision, sampling, faces, 5) for _ in range(2))
    cells = shape[0]*shape[1]
    points = [(k % 2 == 1, 3*((37*k) % cells)+k % 3) for k in range(15)]+[(True, 3*cells-1)]
    for run in (block, single):
        run.steps = sum(counts)-1          # the last step lies past the trace rows
        run.set_trace_points(points)
    assert block.flat()
    for t in block.flat_set:
        t.fill_(float('nan'))              # its contents do not matter
    for count in counts:
        block.block(count)
        for _ in range(count):
            single.step()
    torch.cuda.synchronize()
    assert block.counter.item() == single.counter.item() == sum(counts)
    assert torch.equal(block.traces, single.traces)
    for a, b in zip(state(block), state(single)):
        assert torch.equal(a, b)


def test_grids_that_keep_single_steps(gpu):
    assert not stepper((12, 12, 11), 'float32', 'cell', {}, 1).flat()
    run = stepper((12, 12, 1), 'float32', 'cell', {}, 1)
    run.set_trace_points([(False, k) for k in range(17)])
    assert not run.flat()


def test_graph_of_blocks_follows_eager_steps(gpu):
    """Replays of a captured block with single steps in between."""
    from torchfdtd_amd.graphs import StepGraphs
    block, single = (stepper((50, 40, 1), 'float32', 'cell', {}, 9) for _ in range(2))
    assert block.flat()
    graphs = StepGraphs(block.step, block.states(), 20, 10, block=block.block)
    for run in (single,):
        for t in run.states():
            t.zero_()
    for advance in (10, 1, 10, 10):
        graphs.replay(advance)
        torch.cuda.synchronize()
        for _ in range(advance):
            single.step()
        for a, b in zip(block.states(), single.states()):
            assert torch.equal(a, b)
