"""Blocks of two steps gain nothing from resident groups: the cohort takes them whole."""
import pytest

from test_resident_groups import cohort


@pytest.mark.gpu
def test_blocks_of_two_steps_stay_whole(gpu, monkeypatch):
    from torchfdtd_amd import batch
    whole = cohort('float32')
    for _ in range(5):
        whole.step()
    monkeypatch.setattr(batch, 'WHOLE_BYTES', 0)
    monkeypatch.setattr(batch, 'GROUP_BYTES', 1 << 20)
    grouped = cohort('float32')
    assert len(grouped.groups) > 1
    step, calls = grouped.step, []
    monkeypatch.setattr(grouped, 'step', lambda: (calls.append(1), step()))
    grouped.step_block(2)
    assert len(calls) == 2
    grouped.step_block(3)
    assert len(calls) == 2 and grouped.digest() == whole.digest()
