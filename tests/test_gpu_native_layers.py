"""The native host path of the layers (csrc/torch_ext/ldist_layers.cpp) against the Python route: both make the same
calls of the same library, so outputs, gradients, running means and parameters must agree bit for bit (one-pass p-norm
weight gradients, which collect float atomics, to float32 rounding)."""
import math

import pytest
import torch

import __graft_entry__ as entry
from helpers import gen

pkg = entry.load_package()
cpp = pkg.norm_dist_cpp
pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
INF = float("inf")


@pytest.fixture()
def both_routes():
    """Runs a function on the native path and on the Python route and returns both results."""
    def run(fn):
        try:
            cpp.use_native_layers(True)
            native = fn()
            cpp.use_native_layers(False)
            return native, fn()
        finally:
            cpp.use_native_layers(True)
    return run


def _same(a, b, exact=True):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        if x is not None:
            assert x.shape == y.shape
            assert torch.equal(x, y) if exact else torch.allclose(x, y, rtol=1e-5, atol=1e-5)


# fully connected 2-D, 1x1 image, 3x3 image (image kernels), 5x5 (columns), 3x3 with two positions per row, groups
LAYERS = [dict(kind="fc", cin=37, cout=22), dict(kind="fc", cin=64, cout=9), dict(kind="conv", cin=6, cout=10, k=1, hw=5),
          dict(kind="conv", cin=8, cout=40, k=3, hw=9, group=2), dict(kind="conv", cin=3, cout=32, k=5, hw=8, stride=2)]


@pytest.mark.parametrize("p", [INF, 8.0, 37.3])
@pytest.mark.parametrize("shift,bias", [(True, False), (False, True), (True, True), (False, False)])
@pytest.mark.parametrize("case", range(len(LAYERS)))
def test_layer_routes_agree(both_routes, case, shift, bias, p):
    c = LAYERS[case]
    g = gen(500 + case)
    if c["kind"] == "fc":
        layer = pkg.NormDist(c["cin"], c["cout"], p=p, bias=bias, mean_normalize=shift)
        x = torch.rand(13, c["cin"], generator=g)
    else:
        layer = pkg.NormDistConv(c["cin"], c["cout"], c["k"], stride=c.get("stride", 1), padding=c["k"] // 2, p=p,
                                 group=c.get("group", 1), bias=bias, mean_normalize=shift)
        x = torch.rand(5, c["cin"], c["hw"], c["hw"] + 1, generator=g)
    with torch.no_grad():
        layer.weight.copy_(torch.randn(layer.weight.shape, generator=g) * 0.3)
        if bias:
            layer.bias.copy_(torch.randn(c["cout"], generator=g))
    layer = layer.to(DEV)
    x = x.to(DEV)

    def step(train, grad):
        if shift:
            layer.normalize.running_mean.copy_(torch.linspace(-1, 1, c["cout"], device=DEV))
        layer.train(train)
        for prm in layer.parameters():
            prm.grad = None
        xi = x.clone().requires_grad_(grad)
        with torch.set_grad_enabled(grad):
            y = layer(xi)[0]
        if grad:
            y.backward(torch.sin(torch.arange(y.numel(), device=DEV, dtype=torch.float32)).view_as(y))
        extra = [prm.grad for prm in layer.parameters()] if grad else []
        return [y.detach(), xi.grad, layer.normalize.running_mean.clone() if shift else None] + extra, dict(layer.last_route)

    for train, grad in ((True, True), (False, True), (False, False)):
        (a, ra), (b, rb) = both_routes(lambda: step(train, grad))
        _same(a, b, exact=math.isinf(p))   # finite p without gradients may sum in another order
        assert ra == rb
    if math.isinf(p):
        with torch.no_grad():
            layer.eval()
            (a, ra), (b, rb) = both_routes(lambda: (layer(x, x - 0.1, x + 0.1), dict(layer.last_route)))
        _same(a, b)
        assert ra == rb


def test_a_hooked_mean_shift_is_still_called():
    layer = pkg.NormDist(12, 8, p=INF, bias=False, mean_normalize=True).to(DEV).train()
    seen = []
    handle = layer.normalize.register_forward_hook(lambda mod, args, out: seen.append(out.shape))
    x = torch.rand(4, 12, device=DEV)
    hooked = layer(x)[0]
    handle.remove()
    assert len(seen) == 1 and torch.equal(hooked, layer(x)[0]) and len(seen) == 1


@pytest.mark.parametrize("shape,L", [((3, 5), 1), ((7, 8), 1), ((2, 3), 6), ((2, 3), 7), ((1, 1), 4), ((65, 260), 1)])
def test_evaluation_shift_against_torch(shape, L):
    B, C = shape
    x = torch.randn(B, C, L, generator=gen(3)).to(DEV)
    mean, bias = torch.randn(C, generator=gen(4)).to(DEV), torch.randn(C, generator=gen(5)).to(DEV)
    layer = pkg.NormDistConv(4, C, 1, p=INF, bias=True, mean_normalize=True).to(DEV).eval()
    with torch.no_grad():
        layer.bias.copy_(bias)
        layer.normalize.running_mean.copy_(mean)
        img = torch.rand(B, 4, 1, L, generator=gen(6)).to(DEV)
        y = layer(img)[0]
        raw = pkg.norm_dist(img.view(B, 4, L), layer.weight.view(C, 4), 1, INF)
    assert torch.equal(y.view(B, C, L), (raw - mean.view(1, -1, 1)) + bias.view(1, -1, 1))


def test_margins_and_their_gradients(both_routes):
    lo, up = torch.randn(7, 10, generator=gen(8)).to(DEV), torch.randn(7, 10, generator=gen(9)).to(DEV)
    t = torch.randint(0, 10, (7,), generator=gen(10)).to(DEV)

    def run():
        a, b = lo.clone().requires_grad_(), up.clone().requires_grad_()
        m = pkg.BoundFinalIdentity()(lo, a, b, t)[1]
        m.backward(torch.cos(torch.arange(70, device=DEV, dtype=torch.float32)).view(7, 10))
        return [m.detach(), b.grad], a.grad
    (x, ga), (y, gb) = both_routes(run)
    _same(x, y)
    torch.testing.assert_close(ga, gb, rtol=1e-6, atol=1e-6)


def test_margins_look_the_label_up_as_torch_does(both_routes):
    """What torch's gather does with a target that is no class, both routes do: it sees the targets on either."""
    from torch.utils._python_dispatch import TorchDispatchMode
    up, t = torch.randn(5, 10, generator=gen(8)).to(DEV), torch.arange(5, device=DEV)

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if func is torch.ops.aten.gather.default:
                self.indices.append(args[2].flatten().clone())
            return func(*args, **(kwargs or {}))

    def run():
        mode = Seen()
        mode.indices = []
        with mode:
            pkg.BoundFinalIdentity()(up, up - 1, up + 1, t)
        return mode.indices
    for indices in both_routes(run):
        assert len(indices) == 1 and torch.equal(indices[0], t)


def test_attack_and_optimizer_agree(both_routes):
    def run():
        torch.manual_seed(0)
        net = pkg.Model(pkg.MLP(depth=3, width=1, input_dim=(1, 9, 7)), pkg.BoundFinalIdentity(), 0.1)
        pkg.set_p_norm(net, INF)
        net = net.to(DEV)
        x, t = torch.rand(6, 1, 9, 7, generator=gen(11)).to(DEV), torch.arange(6, device=DEV)
        adv = pkg.AttackPGD(net.eval(), 0.1, 0.03, 3, 1.0, 0.0, random_start=False).find(x, t)
        opt = pkg.AdamW(net, lr=1e-2, weight_decay=1e-2)
        got = [pkg.train_step(net, lambda o, w, t: torch.nn.functional.cross_entropy(o, t), opt, x, t) for _ in range(2)]
        return [adv, torch.tensor(got)] + [prm.detach() for prm in net.parameters()] + list(net.buffers())
    a, b = both_routes(run)
    _same(a, b)


def test_a_layer_refuses_an_input_of_other_channels_than_its_weight():
    for k, c in ((3, 12), (3, 4), (1, 12), (1, 4)):
        layer = pkg.NormDistConv(8, 8, k, padding=k // 2, p=INF, bias=False).to(DEV).eval()
        x = torch.rand(2, c, 6, 6, device=DEV)
        for p in (INF, 8.0):
            layer.p = p
            with pytest.raises((RuntimeError, AssertionError)):
                layer(x)
        layer.p = INF
        with torch.no_grad(), pytest.raises((RuntimeError, AssertionError)):
            layer(x, x, x)


def test_vectors_that_are_not_one_value_per_channel_take_the_python_route(both_routes):
    layer = pkg.NormDist(12, 8, p=INF, bias=True, mean_normalize=True).to(DEV).eval()
    layer.bias = torch.nn.Parameter(torch.tensor([0.75], device=DEV))            # broadcasts over the channels
    layer.normalize.running_mean = torch.arange(16.0, device=DEV)[::2]          # strided
    x = torch.rand(4, 12, generator=gen(12)).to(DEV)
    a, b = both_routes(lambda: [t.detach() for t in layer(x, x - 0.1, x + 0.1)])
    _same(a, b)


def test_bounds_carry_the_gradient_of_the_bias(both_routes):
    layer = pkg.NormDist(12, 8, p=INF, bias=True).to(DEV).eval()
    x = torch.rand(4, 12, generator=gen(13)).to(DEV)

    def run():
        layer.bias.grad = None
        y, lo, hi = layer(x, x - 0.1, x + 0.1)
        (2 * lo.sum() + 3 * hi.sum()).backward()
        return [y.detach(), lo.detach(), hi.detach(), layer.bias.grad]
    a, b = both_routes(run)
    _same(a, b)
    assert torch.equal(a[3], torch.full((8,), 20.0, device=DEV))


def test_transformations_see_every_operation():
    import torch.autograd.forward_ad as fwd
    layer = pkg.NormDist(12, 8, p=8.0, bias=False).to(DEV)
    for prm in layer.parameters():
        prm.requires_grad_(False)
    x = torch.rand(4, 12, device=DEV)
    with fwd.dual_level(), pytest.raises(RuntimeError):        # no forward derivative: refused, not dropped
        layer(fwd.make_dual(x, torch.ones_like(x)))
    lo, up = torch.rand(3, 5, 10, device=DEV), torch.rand(3, 5, 10, device=DEV)
    t = torch.randint(0, 10, (5,), device=DEV)
    margins = pkg.BoundFinalIdentity()
    got = torch.func.vmap(lambda a, b: margins(a, a, b, t)[1])(lo, up)
    assert torch.equal(got, torch.stack([margins(a, a, b, t)[1] for a, b in zip(lo, up)]))


def test_empty_batches_and_other_dimensions():
    none = torch.empty(0, 10, device=DEV)
    assert pkg.BoundFinalIdentity()(none, none, none, torch.empty(0, dtype=torch.int64, device=DEV))[1].shape == (0, 10)
    x, w = torch.rand(4, 12, device=DEV), torch.rand(8, 12, device=DEV)
    with pytest.raises((RuntimeError, IndexError)):
        pkg.norm_dist(x, w, 1, INF)
    with pytest.raises((RuntimeError, IndexError)):
        pkg.norm_dist(x.view(4, 12, 1), w.view(8, 12, 1, 1), 1, INF)


# Small layers whose sums are shared out over workgroups unless asked not to: outputs, rows (300 x 40 -> 24), a window.
@pytest.mark.parametrize("p", [3.0, 8.0, 37.3])
@pytest.mark.parametrize("case", [(64, 512, 1024, 0), (300, 40, 24, 0), (33, 130, 260, 0), (6, 5, 300, 11)])
def test_deterministic_p_norm_gradients(both_routes, case, p):
    B, cin, cout, hw = case
    x = torch.rand(*((B, cin, hw, hw) if hw else (B, cin)), generator=gen(21)).to(DEV)
    layer = pkg.NormDistConv(cin, cout, 3, padding=1, p=p) if hw else pkg.NormDist(cin, cout, p=p)
    layer = layer.to(DEV)

    def run():
        layer.zero_grad()
        xi = x.clone().requires_grad_()
        y = layer(xi)[0]
        y.backward(torch.sin(torch.arange(y.numel(), device=DEV, dtype=torch.float32)).view_as(y))
        return [xi.grad, layer.weight.grad.clone()]
    torch.use_deterministic_algorithms(True)
    try:
        native, python = both_routes(lambda: [run() for _ in range(6)])
    finally:
        torch.use_deterministic_algorithms(False)
    for got in native[1:] + python:
        _same(native[0], got)
    # The shared form: the same sums in another order, of terms that are powers of numbers rounded a few times (p * 2^-23 and a
    # few times that); the terms' signs alternate, which a factor of eight covers.
    for a, b in zip(native[0], run()):
        assert (a - b).norm() <= 8 * 2.0 ** -23 * (p + 2) * b.norm()


@pytest.mark.parametrize("changed", ["host", "strided", "wider type", "shorter"])
@pytest.mark.parametrize("p", [INF, 8.0])
@pytest.mark.parametrize("case", ["fc", "image"])
def test_saved_tensors_that_a_hook_has_changed_are_refused(case, p, changed):
    """What an unpack hook returns is not what was saved: the native nodes say so before a kernel reads it."""
    from gpu_common import say
    say("saved tensors", case, p, changed)
    back = {"host": lambda t: t.cpu(), "wider type": lambda t: t.double(), "shorter": lambda t: t[:-1].contiguous(),
            "strided": lambda t: torch.stack([t, t], -1)[..., 0]}[changed]
    layer = (pkg.NormDist(12, 20, p=p, bias=False) if case == "fc" else
             pkg.NormDistConv(4, 20, 3, padding=1, p=p, bias=False)).to(DEV)
    x = torch.rand(*((6, 12) if case == "fc" else (6, 4, 7, 8)), device=DEV, requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, back):
        y = layer(x)[0]
    with pytest.raises(RuntimeError, match="saved"):
        y.sum().backward()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(DEV)):   # as it was saved: taken
        y = layer(x)[0]
    got = torch.autograd.grad(y.sum(), x)[0]
    _same([got], [torch.autograd.grad(layer(x)[0].sum(), x)[0]], exact=p == INF)
