"""The narrow forward layer on an FP32 input, which it rounds as it reads, against the same input rounded before."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (n, d, h, w, ci, co, ks, stride, pad): at most 32 values of K, rows of one and of several workgroups, every edge.
CASES = [(1, 1, 1, 1, 1, 8, 3, 1, 1), (2, 8, 64, 64, 1, 32, 3, 2, 1), (3, 5, 7, 9, 1, 72, 3, 1, 0), (2, 6, 5, 4, 1, 24, 3, 1, 2),
         (2, 4, 9, 33, 1, 40, 3, 2, 1), (70, 1, 1, 1, 32, 32, 1, 1, 0), (5, 3, 4, 5, 20, 12, 1, 2, 0)]


@pytest.mark.parametrize('n,d,h,w,ci,co,ks,stride,pad', CASES)
def test_wide_source_equals_the_rounded_one(gpu, n, d, h, w, ci, co, ks, stride, pad):
    from torchfdtd_amd.surrogate import _forward, _operands, conv_rows, conv_shape
    gen = torch.Generator(device='cuda').manual_seed(3)
    x = torch.randn((n, d, h, w, ci), device=gpu, generator=gen)
    x.view(-1)[::7] = 1+2.**-8         # halfway between two bf16 values
    if x.numel() > 40:
        x.view(-1)[5], x.view(-1)[31] = float('inf'), float('nan')
    weight = torch.randn((co, ks, ks, ks, ci), device=gpu, generator=gen)
    bias = torch.randn(co, device=gpu, generator=gen)
    shape, _ = conv_shape(tuple(x.shape), ci, co, ks, stride, pad)
    assert shape.kp == 32
    (w16, _, parts), = _operands([shape], [weight], [False])
    results = []
    for source in (x, x.to(torch.bfloat16)):
        out = [torch.empty((conv_rows(shape), co), device=gpu, dtype=t) for t in (torch.float32, torch.float32, torch.bfloat16)]
        _forward(shape, source, w16, parts, bias, True, pre=out[0], y=out[1], act=out[2])
        results.append(out)
    for a, b in zip(*results):
        assert torch.equal(torch.nan_to_num(a, nan=123.), torch.nan_to_num(b, nan=123.))


@pytest.mark.parametrize('channels,batch', [((8,), 1), ((32, 40), 3), ((8,)*7, 2)])
@pytest.mark.parametrize('trained', ['all', 'head', 'none'])
def test_network_equals_its_layers(gpu, channels, batch, trained):
    """The network, whose head shares the trunk's operand launch (not beyond eight layers) and keeps bf16 without a
    backward, against conv3d and linear layer by layer: outputs and gradients equal."""
    from torchfdtd_amd.surrogate import SurrogateNet, conv3d, linear
    net = SurrogateNet(channels=channels, hidden=24, outputs=8, seed=2).to(gpu)
    for p in net.parameters():
        p.requires_grad_(trained == 'all')
    for p in net.head:
        p.requires_grad_(trained != 'none')
    rho = torch.rand((batch, 17, 12, 8), device=gpu, generator=torch.Generator(device='cuda').manual_seed(1))

    def layers():
        x = rho.unsqueeze(-1)
        for w, b in zip(net.weights, net.biases):
            x = conv3d(x, w, b, 2, 1, True)
        return linear(linear(x.mean(dim=(1, 2, 3)), net.head[0], net.head[1]), net.head[2], net.head[3], activation=False)

    wanted = [p for p in net.parameters() if p.requires_grad]
    results = []
    for y in (net(rho), layers()):
        results.append([y.detach(), *(torch.autograd.grad(y.square().sum(), wanted) if wanted else ())])
    for a, b in zip(*results):
        assert torch.equal(a, b)
    with torch.no_grad():
        assert torch.equal(net(rho), results[0][0])
