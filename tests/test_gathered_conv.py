"""The gathered convolution kernels at the edges of their tiles, against FP64 on the same bf16 operands.

Bounds: an FP32 sum of K products of bf16 values (exact in FP32) is off by at most K 2^-24 times the sum
of the products' magnitudes.
"""
import ctypes
import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# Rows of one tile less and more, ragged columns, chunks that straddle taps (channels 8, 24, 40, 72), strided
# parities on odd and even extents, inputs one cell deep, one-channel inputs, linear layers.
LAYERS = [((1, 4, 4, 8), 32, 32, 3, 1, 1), ((2, 5, 7, 9), 64, 72, 3, 1, 1), ((3, 9, 6, 7), 32, 136, 3, 2, 1), ((2, 8, 8, 3), 8, 24, 3, 2, 0),
          ((1, 3, 3, 3), 40, 8, 3, 1, 0), ((5, 7, 1, 1), 72, 64, 3, 2, 1), ((129, 1, 1, 1), 256, 32, 1, 1, 0), ((2, 5, 4, 3), 96, 40, 1, 2, 0),
          ((2, 11, 9, 5), 1, 32, 3, 2, 1), ((1, 6, 5, 4), 1, 70, 3, 1, 1), ((33, 1, 1, 1), 24, 8, 1, 1, 0), ((24, 16, 16, 2), 32, 64, 3, 2, 1)]


def direct(x, w, b, stride, pad):
    return F.conv3d(x.permute(0, 4, 1, 2, 3), w.permute(0, 4, 1, 2, 3), b, stride=stride, padding=pad).permute(0, 2, 3, 4, 1)


@pytest.mark.parametrize('shape,ci,co,ks,stride,pad', LAYERS)
def test_pre_activation_and_gradients_within_the_fp32_bound(gpu, shape, ci, co, ks, stride, pad):
    from torchfdtd_amd.surrogate import _forward, _input_gradient, _layer_gradients, _operands, conv_shape
    gen = torch.Generator().manual_seed(ci*co+ks)
    x, w = torch.randn((*shape, ci), generator=gen).bfloat16(), (torch.randn((co, ks, ks, ks, ci), generator=gen)/math.sqrt(ks**3*ci)).bfloat16()
    b = torch.randn(co, generator=gen)
    s, out = conv_shape((*shape, ci), ci, co, ks, stride, pad)
    m, k = shape[0]*math.prod(out), ks**3*ci
    (w16, wt, parts), = _operands([s], [w.float().cuda()], [True])
    pre = torch.full((m, co), float('nan'), device=gpu)
    act = torch.empty((m, co), device=gpu, dtype=torch.bfloat16)
    _forward(s, x.cuda(), w16, parts, b.cuda(), False, pre=pre, act=act)
    xd, wd, bd = x.double().requires_grad_(True), w.double().requires_grad_(True), b.double()
    expected = direct(xd, wd, bd, stride, pad).reshape(m, co)
    magnitude = direct(x.double().abs(), w.double().abs(), bd.abs(), stride, pad).reshape(m, co)
    assert bool(((pre.cpu().double()-expected).abs() <= (k+1)*2**-24*magnitude).all())
    assert torch.equal(act.cpu(), pre.cpu().bfloat16())
    if co % 8:
        return
    dy = torch.randn((m, co), generator=gen).bfloat16()
    dpre16, dw, grad_bias = _layer_gradients(s, dy.float().cuda(), pre, 0, x.cuda())
    assert torch.equal(dpre16.cpu(), dy)
    dx = _input_gradient(s, dpre16, w16, wt, parts)
    want_x, want_w = torch.autograd.grad(expected, (xd, wd), dy.double())
    xa, wa = x.double().abs().requires_grad_(True), w.double().abs().requires_grad_(True)
    size_x, size_w = torch.autograd.grad(direct(xa, wa, None, stride, pad).reshape(m, co), (xa, wa), dy.double().abs())
    dw = dw.cpu()[:, :k].reshape(w.shape).double()
    assert bool(((dw-want_w).abs() <= (m+1)*2**-24*size_w).all())
    assert bool(((dx.cpu().double().reshape(want_x.shape)-want_x).abs() <= (ks**3*co+1)*2**-24*size_x).all())
    assert bool(((grad_bias.cpu().double()-dy.double().sum(0)).abs() <= (m+1)*2**-24*dy.double().abs().sum(0)).all())


def test_taps_in_the_padding_keep_what_infinite_weights_give(gpu):
    """A tap that lies in the padding for every row adds 0 * w: nothing for finite weights, NaN for an infinite one."""
    from torchfdtd_amd.surrogate import conv3d
    x = torch.ones((2, 1, 6, 6, 32), device=gpu)
    w = torch.full((32, 3, 3, 3, 32), .5, device=gpu)
    b = torch.zeros(32, device=gpu)
    assert torch.isfinite(conv3d(x, w, b, 1, 1, False)).all()
    w[5, 0, 1, 1, 7] = float('inf')
    y = conv3d(x, w, b, 1, 1, False)
    assert torch.isnan(y[..., 5]).all()
    assert torch.isfinite(y[..., :5]).all() and torch.isfinite(y[..., 6:]).all()


def test_network_equals_its_layers_one_by_one(gpu):
    """The network's trunk against conv3d after conv3d: the same operations, so equal outputs and gradients."""
    from torchfdtd_amd.surrogate import SurrogateNet, conv3d, linear
    net = SurrogateNet(channels=(32, 40, 64), hidden=24, outputs=8, seed=4).to(gpu)
    gen = torch.Generator().manual_seed(9)
    rho = torch.rand((3, 18, 13, 9), generator=gen).to(gpu).requires_grad_(True)
    x = rho.unsqueeze(-1)
    for w, b in zip(net.weights, net.biases):
        x = conv3d(x, w, b, stride=2, pad=1, activation=True)
    x = linear(x.mean(dim=(1, 2, 3)), net.head[0], net.head[1])
    expected = linear(x, net.head[2], net.head[3], activation=False)
    parameters = [rho, *net.parameters()]
    want = torch.autograd.grad(expected.square().sum(), parameters)
    got = net(rho)
    assert torch.equal(got, expected)
    for a, b in zip(torch.autograd.grad(got.square().sum(), parameters), want):
        assert torch.equal(a, b)
    with torch.no_grad():
        assert torch.equal(net(rho), expected)


@pytest.mark.parametrize('ci,co,ks', [(1, 6, 1), (5, 32, 1), (31, 36, 1), (32, 64, 1), (1, 33, 3)])
def test_narrow_layers_find_their_taps_and_round_as_torch(gpu, ci, co, ks):
    """At most 32 values of K, split into taps and channels; bf16 values of ties, overflow, infinities and NaN."""
    from torchfdtd_amd.surrogate import _forward, _operands, conv_shape
    gen = torch.Generator().manual_seed(ci+co)
    shape = (3, 5, 4, 7)
    x, w = torch.randn((*shape, ci), generator=gen).bfloat16(), torch.randn((co, ks, ks, ks, ci), generator=gen).bfloat16()
    b = torch.randn(co, generator=gen)
    b[:5] = torch.tensor([math.inf, -math.inf, math.nan, 3.4e38, 1+2**-8])
    s, out = conv_shape((*shape, ci), ci, co, ks, 1, ks // 2)
    m, k = shape[0]*math.prod(out), ks**3*ci
    (w16, _, parts), = _operands([s], [w.float().cuda()], [False])
    pre, act = torch.empty((m, co), device=gpu), torch.empty((m, co), device=gpu, dtype=torch.bfloat16)
    _forward(s, x.cuda(), w16, parts, b.cuda(), False, pre=pre, act=act)
    expected = direct(x.double(), w.double(), b.double(), 1, ks // 2).reshape(m, co)
    magnitude = direct(x.double().abs(), w.double().abs(), b.double().abs(), 1, ks // 2).reshape(m, co)
    got = pre.cpu().double()
    assert bool(((got-expected).abs() <= (k+1)*2**-24*magnitude)[:, 3:].all())
    assert torch.equal(got[:, :2], expected[:, :2]) and bool(got[:, 2].isnan().all())
    assert torch.equal(act.cpu().nan_to_num(7.), pre.cpu().bfloat16().nan_to_num(7.))
    assert torch.equal(act.cpu().isnan(), pre.cpu().isnan())


@pytest.mark.parametrize('shape,ci,co,ks,stride,pad', [((9, 2, 3, 2), 64, 72, 3, 1, 1), ((40, 3, 2, 5), 8, 64, 3, 2, 1), ((2, 17, 13, 11), 32, 32, 3, 2, 0),
                                                       ((70, 1, 2, 1), 16, 136, 3, 1, 1), ((3, 1, 1, 65), 40, 24, 1, 2, 0), ((1, 66, 1, 1), 24, 64, 3, 1, 1),
                                                       ((2, 64, 4, 3), 8, 32, 3, 1, 0), ((5, 3, 64, 3), 16, 128, 3, 1, 1)])
def test_weight_gradient_walks_every_position(gpu, shape, ci, co, ks, stride, pad):
    """Positions move on by 64 with carries: axes of 1 to 66, several samples a stage, ends inside a stage, splits."""
    from torchfdtd_amd.surrogate import _layer_gradients, conv_shape
    s, out = conv_shape((*shape, ci), ci, co, ks, stride, pad)
    gen = torch.Generator().manual_seed(ci+co)
    m, k = shape[0]*math.prod(out), ks**3*ci
    x, dy = torch.randn((*shape, ci), generator=gen).bfloat16(), torch.randn((m, co), generator=gen).bfloat16()
    _, dw, _ = _layer_gradients(s, dy.float().cuda(), torch.zeros((m, co), device=gpu), 0, x.cuda())

    def direct_gradient(a, b):
        w = torch.zeros((co, ks, ks, ks, ci), dtype=torch.float64, requires_grad=True)
        return torch.autograd.grad(direct(a, w, None, stride, pad).reshape(m, co), w, b)[0]
    want, size = direct_gradient(x.double(), dy.double()), direct_gradient(x.double().abs(), dy.double().abs())
    assert bool(((dw.cpu()[:, :k].reshape(want.shape).double()-want).abs() <= (m+1)*2**-24*size).all())
