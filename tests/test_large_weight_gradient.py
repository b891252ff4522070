"""The weight gradient of a layer of 2^30 weights: its splits' sum takes more values than one launch has lanes for."""
import ctypes

import pytest
import torch

from torchfdtd_amd import _native as N


@pytest.mark.gpu
def test_gradient_of_a_gigaweight_linear_layer(gpu):
    from torchfdtd_amd.surrogate import ConvShape
    lib, rows, width = N.library(), 8, 32768
    shape = ConvShape(rows, 1, 1, 1, width, width, 1, 1, 0, width)
    gen = torch.Generator(device='cuda').manual_seed(3)
    x, dy = (torch.randint(-4, 5, (rows, width), device='cuda', generator=gen).to(torch.bfloat16) for _ in range(2))
    splits = lib.tfdtd_conv_wgrad_splits(ctypes.byref(shape))
    partial = torch.empty((splits, width, width), device='cuda')
    dw = torch.full((width, width), float('nan'), device='cuda')
    N.check(lib.tfdtd_conv_wgrad_rows(ctypes.byref(shape), dy.data_ptr(), x.data_ptr(), partial.data_ptr(), dw.data_ptr(),
                                      N.stream_handle()), 'wgrad')
    # Small whole numbers: every sum is exact.
    for o in range(0, width, 4096):
        assert torch.equal(dw[o:o+4096], dy[:, o:o+4096].float().t().contiguous()@x.float())
