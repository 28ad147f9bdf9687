"""Layers in evaluation mode: the forward kernels apply the running mean and the bias on their way out.  Against the operator
without them followed by torch's subtraction and addition, bit for bit, on a size of every kernel."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

INF = float("inf")
FC = [  # batch, inputs, outputs: few rows, small tiles, the large tiles, few outputs, lists of outermost values
    (1, 75, 22), (2, 1024, 1025), (3, 300, 130), (7, 129, 64), (100, 1024, 1024), (60, 515, 77), (512, 784, 5120), (1030, 100, 200),
    (9, 512, 10), (1, 5120, 10), (1024, 2048, 2048), (130, 1000, 5121),
]


def build(layer, bias, mean):
    from gpu_common import DEV
    layer = layer.to(DEV).eval()
    g = torch.Generator(device=DEV).manual_seed(5)
    with torch.no_grad():
        layer.weight.normal_(0, 1 / math.sqrt(layer.weight[0].numel()), generator=g)
        if bias:
            layer.bias.normal_(0, 1, generator=g)
        if mean:
            layer.normalize.running_mean.normal_(0, 1, generator=g)
    return layer, g


def expected(layer, raw):
    shape = (1, -1) + (1,) * (raw.dim() - 2)
    if layer.normalize is not None:
        raw = raw - layer.normalize.running_mean.view(shape)
    return raw if layer.bias is None else raw + layer.bias.detach().view(shape)


@pytest.mark.parametrize("bias,mean", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("p", [INF, 8.0, 20.5])
@pytest.mark.parametrize("case", FC)
def test_fully_connected(case, p, bias, mean):
    from gpu_common import DEV, pkg, say
    B, K, N = case
    say("shifted fc", case, p, bias, mean)
    layer, g = build(pkg.NormDist(K, N, p=p, bias=bias, mean_normalize=mean), bias, mean)
    x = torch.rand(B, K, device=DEV, generator=g)
    w = layer.weight.detach().view(N, K)
    with torch.no_grad():
        raw = pkg.norm_dist(x.view(B, K, 1), w, 1, p).view(B, N)
        assert torch.equal(layer(x)[0], expected(layer, raw))
    if not math.isinf(p):
        return
    xg = x.clone().requires_grad_(True)   # with positions
    y = layer(xg)[0]
    assert torch.equal(y.detach(), expected(layer, raw))
    up = torch.randn(B, N, device=DEV, generator=g)
    y.backward(up)
    xr = x.clone().requires_grad_(True)
    pkg.norm_dist(xr.view(B, K, 1), w, 1, p).backward(up.view(B, N, 1))
    assert torch.equal(xg.grad, xr.grad)
    if bias:
        torch.testing.assert_close(layer.bias.grad, up.sum(0))
    with torch.no_grad():
        lo, hi = x - 0.05, x + 0.05
        rl, ru = pkg.inf_dist_bound(lo.view(B, K, 1), hi.view(B, K, 1), w, 1)
        _, ol, ou = layer(x, lo, hi)
        assert torch.equal(ol, expected(layer, rl.view(B, N))) and torch.equal(ou, expected(layer, ru.view(B, N)))


@pytest.mark.parametrize("case", [(3, 32, 14, 14, 64, 1, 1), (2, 8, 16, 16, 24, 2, 1), (2, 16, 9, 11, 10, 1, 2), (40, 32, 32, 32, 32, 1, 1)])
def test_images(case):
    from gpu_common import DEV, cpp, pkg, say
    B, C, H, W, CO, G, s_ = case
    say("shifted image", case)
    layer, g = build(pkg.NormDistConv(C, CO, 3, stride=s_, padding=1, group=G, p=INF, bias=True, mean_normalize=True), True, True)
    x = torch.rand(B, C, H, W, device=DEV, generator=g)
    lo, hi = x - 0.05, x + 0.05
    w = layer.weight.detach().view(CO, -1)
    ho, wo = (H - 1) // s_ + 1, (W - 1) // s_ + 1
    columns = lambda t: torch.nn.functional.unfold(t, 3, 1, 1, s_)
    with torch.no_grad():
        raw = pkg.norm_dist(columns(x), w, G, INF).view(B, CO, ho, wo)
        rl, ru = (t.view(B, CO, ho, wo) for t in pkg.inf_dist_bound(columns(lo), columns(hi), w, G))
        y, ol, ou = layer(x, lo, hi)
    assert torch.equal(y, expected(layer, raw))
    assert torch.equal(ol, expected(layer, rl)) and torch.equal(ou, expected(layer, ru))
    y = layer(x.clone().requires_grad_(True))[0]
    assert torch.equal(y.detach(), expected(layer, raw))
