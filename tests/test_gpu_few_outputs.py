"""Fully connected layers of few outputs: both p-norm gradients in one launch, and the forward passes of one and two rows."""
import pytest
import torch

import oracle
from helpers import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [2.0, 3.0, 4.0, 8.0, 1.7, 37.3, 100.0])
@pytest.mark.parametrize("case", [(1, 1, 64, 10), (9, 1, 75, 5), (64, 1, 512, 10), (65, 1, 130, 16), (200, 3, 65, 12), (515, 1, 1030, 9), (3, 2, 9, 1)])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** 14])   # outputs inside and outside the range of the factored form
def test_both_gradients(case, p, scale):
    from gpu_common import DEV, cpp, say
    B, G, K, NG = case
    say("few outputs backward", case, p, scale)
    x = torch.randn(B, G * K, 1, generator=gen(91)) * scale
    w = torch.randn(G * NG, K, generator=gen(92)) * scale
    go = torch.randn(B, G * NG, 1, generator=gen(93))
    base = torch.randn(G * NG, K, generator=gen(94))
    xd, wd = x.double().view(B, G, 1, K), w.double().view(1, G, NG, K)
    df = xd - wd
    out = df.abs().amax(-1) * (df.abs() / df.abs().amax(-1, keepdim=True)).pow(p).sum(-1).pow(1 / p)   # (B, G, NG)
    out = out.float()
    t = go.double().view(B, G, NG, 1) * (df.abs() / out.double().unsqueeze(-1)).pow(p - 1) * df.sign()
    gi, gw = t.sum(2), base.double().view(G, NG, K) - t.sum(0)
    # Relative error of a term in units of 2^-24: the difference, the reciprocal and their product are off by 4, the logarithm by
    # as much as 1 near u = 1, all p - 1 times in the power; with L = (p-1) log2 u, the logarithm's unit in the last place and the
    # product's rounding are 3 |L| ln 2 of the power, exponential and factor 4.  Then one rounding per addition.
    log = ((p - 1) * (df.abs() / out.double().unsqueeze(-1)).log2()).abs().clamp(max=200)
    size = t.abs() * (5 * p + 2.1 * log + 4) * 2.0 ** -24
    bound_i = size.sum(2) + NG * 2.0 ** -24 * t.abs().sum(2) + 1e-37
    bound_w = size.sum(0) + 80 * 2.0 ** -24 * (t.abs().sum(0) + base.double().view(G, NG, K).abs())
    di = torch.full((B, G * K, 1), float("nan"), device=DEV)
    dw = base.to(DEV).clone()
    cpp.norm_dist_backward(go.to(DEV), x.to(DEV), w.to(DEV), out.view(B, G * NG, 1).to(DEV), di, dw, G, p)
    torch.cuda.synchronize()
    assert ((di.cpu().double().view(B, G, K) - gi).abs() <= bound_i).all()
    assert ((dw.cpu().double().view(G, NG, K) - gw).abs() <= bound_w).all()


@pytest.mark.parametrize("case", [(1, 2048, 10), (2, 5120, 10), (1, 1027, 16), (2, 1030, 3), (3, 2052, 7)])
def test_forward_of_a_long_reduction_bit_exact(case):
    from gpu_common import DEV, gpu_inf_forward, gpu_value_bound_forward, say
    B, K, N = case
    say("few outputs forward", case)
    x = (torch.randn(B, K, 1, generator=gen(95)) * 8).round() / 8     # ties
    w = (torch.randn(N, K, generator=gen(96)) * 8).round() / 8
    eo, ep = oracle.inf_dist_forward(x, w, 1)
    out, pos = gpu_inf_forward(x, w, 1)
    assert torch.equal(out, eo) and torch.equal(pos, ep)
    lo, up = x - 0.25, x + 0.25
    lo[0, 5], up[-1, K - 1] = float("nan"), float("inf")
    el, eu = oracle.inf_dist_bound_forward(lo, up, w, 1)
    v, ol, ou = gpu_value_bound_forward(x, lo, up, w, 1)
    assert torch.equal(v, eo)
    assert torch.equal(torch.nan_to_num(ol, nan=-7.0), torch.nan_to_num(el, nan=-7.0))
    assert torch.equal(torch.nan_to_num(ou, nan=-7.0), torch.nan_to_num(eu, nan=-7.0))


@pytest.mark.parametrize("p", [3.0, 8.0, 37.3])
@pytest.mark.parametrize("case", [(1, 5120, 10), (2, 1030, 3), (1, 1027, 16)])
def test_values_of_one_and_two_rows(case, p):
    from gpu_common import DEV, cpp, say
    B, K, N = case
    say("few outputs values", case, p)
    x, w = torch.randn(B, K, 1, generator=gen(97)), torch.randn(N, K, generator=gen(98))
    out = torch.full((B, N, 1), float("nan"), device=DEV)
    cpp.norm_dist_forward_values(x.to(DEV), w.to(DEV), out, 1, p)
    df = (x.double().view(B, 1, K) - w.double()).abs()
    exact = df.amax(-1) * (df / df.amax(-1, keepdim=True)).pow(p).sum(-1).pow(1 / p)
    # a term is off by p + 45 units at the most, which the root divides by p; root and scale add a few
    torch.testing.assert_close(out.cpu().double().view(B, N), exact, rtol=((p + 45) / p + 20) * 2.0 ** -23, atol=0.0)


@pytest.mark.parametrize("p", [2.0, 37.3])
def test_both_gradients_of_as_many_rows_as_an_index_counts(p):
    """One input, one output, 2^31 - 100 rows: counting rows past the last of them in 32 bits with a sign would start over."""
    from gpu_common import DEV, cpp, say
    B = 2 ** 31 - 100
    say("few outputs backward, rows", B, p)
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("48 GiB of device memory")
    x, out = torch.full((B, 1, 1), 0.5, device=DEV), torch.full((B, 1, 1), 0.5, device=DEV)
    go, gi = torch.zeros(B, 1, 1, device=DEV), torch.full((B, 1, 1), float("nan"), device=DEV)
    rows = torch.tensor([0, 63, 64, B // 2, 2 ** 31 - 2 ** 21 - 1, 2 ** 31 - 2 ** 21, B - 2 ** 20, B - 65, B - 2, B - 1], device=DEV)
    signs = torch.tensor([1.0, -1.0], device=DEV).repeat(5)
    x[rows, 0, 0] = 0.5 * signs
    go[rows, 0, 0] = 2.0 ** torch.arange(10, device=DEV)
    gw = torch.zeros(1, 1, device=DEV)
    cpp.norm_dist_backward(go, x, torch.zeros(1, 1, device=DEV), out, gi, gw, 1, p)   # |x - w| = out: the powers are one
    assert gw.item() == -(go[rows, 0, 0] * signs).sum().item()
    assert torch.equal(gi[rows, 0, 0], go[rows, 0, 0] * signs)
    gi[rows, 0, 0] = 0.0
    assert not any(part.any().item() for part in gi.view(-1).split(2 ** 28))      # NaN counts as true
