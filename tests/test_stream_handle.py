"""The stream handle of a device that is no GPU is refused before anything else (CPU)."""
import pytest
import torch

from torchfdtd_amd import _native as N


@pytest.mark.parametrize('device', ['cpu', torch.device('cpu'), torch.device('meta')])
def test_a_device_without_streams_is_refused(device):
    with pytest.raises(ValueError, match='Expected a cuda device'):
        N.stream_handle(device)
