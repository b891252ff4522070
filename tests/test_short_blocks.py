"""Blocks of two and three steps: a large flat grid takes them as half steps, bit for bit what single steps give.

Patches write the second buffer set, half steps leave it as it was.
"""
import pytest
import torch

from test_plane_march import state, stepper

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape,precision,count,patches', [
    ((448, 448, 1), 'float32', 2, True), ((449, 448, 1), 'float32', 2, False), ((449, 448, 1), 'float32', 3, True),
    ((449, 448, 1), 'float64', 3, False), ((449, 448, 1), 'float64', 4, True), ((448, 448, 1), 'float64', 2, True),
    ((900, 800, 1), 'float64', 3, True), ((900, 800, 1), 'float64', 2, False)])
def test_short_blocks(gpu, shape, precision, count, patches):
    block, single = (stepper(shape, precision, 'cell', {}, 4) for _ in range(2))
    for run in (block, single):
        run.set_trace_points([(False, 3*777+2), (True, 3*shape[0]*shape[1]-1)])
    assert block.flat()
    for t in block.flat_set:
        t.fill_(float('nan'))
    block.block(count)
    for _ in range(count):
        single.step()
    torch.cuda.synchronize()
    assert bool(block.flat_set[0].isnan().all()) != patches
    assert block.counter.item() == single.counter.item() == count
    assert torch.equal(block.traces, single.traces)
    for a, b in zip(state(block), state(single)):
        assert torch.equal(a, b)
