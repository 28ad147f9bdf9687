"""The native host path of the layers (csrc/torch_ext/ldist_layers.cpp) where no GPU is needed: what it does before it looks at
the device of its tensors."""
import threading
import time
from unittest import mock

import numpy as np
import pytest
import torch

import __graft_entry__ as entry

pkg = entry.load_package()


@pytest.fixture(scope="module")
def ops():
    module = pkg.norm_dist_cpp._compiled("ldist_layers")
    if module is None:
        pytest.skip("torch_ext has not been built")
    return module


def _longest_pause_of_another_thread(call):
    """Seconds of `call`, and the longest time another thread found no turn meanwhile."""
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)
    other = threading.Thread(target=tick)
    other.start()
    time.sleep(0.02)
    begin = time.perf_counter()
    with pytest.raises(RuntimeError, match="CUDA"):
        call()
    end = time.perf_counter()
    stop.set()
    other.join()
    inside = [begin] + [t for t in ticks if begin < t < end] + [end]
    return end - begin, max(b - a for a, b in zip(inside, inside[1:]))


def test_other_threads_run_during_a_call(ops):
    """The functions make strided tensors contiguous before they refuse what is not on a GPU: time to spend without the
    interpreter lock.  Held, no other thread would have a turn before the call returns."""
    wide = torch.zeros(6000, 6000).t()
    targets = torch.zeros(6000, dtype=torch.int64)
    threads = torch.get_num_threads()
    torch.set_num_threads(1)
    try:
        for call in (lambda: ops.pgd_step(wide, wide, wide, 0.1, 0.1, 0.0, 1.0), lambda: ops.margins(wide, wide, targets),
                     lambda: ops.layer(wide, wide.view(6000, 6000, 1, 1), None, None, 0.0, False, 1, 8.0, 1, 1, 0, 1, True, 0)):
            took, pause = _longest_pause_of_another_thread(call)
            assert pause < 0.5 * took, (took, pause)
    finally:
        torch.set_num_threads(threads)


@pytest.mark.parametrize("stride,padding,dilation", [(0, 1, 1), (-1, 1, 1), (1, -1, 1), (1, 1, 0)])
def test_a_window_that_is_none_is_refused_with_an_exception(ops, stride, padding, dilation):
    """A stride of zero would divide the process away, on whatever device the tensors are."""
    x, w = torch.zeros(2, 3, 8, 8), torch.zeros(4, 3, 3, 3)
    for call in (lambda: ops.layer(x, w, None, None, 0.0, False, 1, 8.0, 3, stride, padding, dilation, True, 0),
                 lambda: ops.layer_bounds(x, x, w, None, None, 1, 3, stride, padding, dilation)):
        with pytest.raises(RuntimeError, match="window"):
            call()


@pytest.mark.parametrize("weight", [(8, 12, 1, 1), (8, 3, 2, 2), (8, 12, 1), (96,)])
def test_weights_that_are_no_matrix_are_refused(ops, weight):
    """As the entry points of the library's torch extension do, whatever the weight's values would make of it."""
    x, w = torch.zeros(4, 12, 5), torch.zeros(weight)
    for call in (lambda: ops.norm_dist(x, w, 1, 8.0), lambda: ops.inf_dist_bound(x, x, w, 1)):
        with pytest.raises(RuntimeError, match="weight 2-D"):
            call()


def test_adamw_takes_any_number_as_a_step_or_rate(ops, monkeypatch):
    """A restored state may hold the step count as a float or a tensor; a rate may be a tensor."""
    layer = pkg.NormDist(6, 4, p=8.0)
    opt = pkg.AdamW(layer, lr=torch.tensor(1e-2))
    for prm in layer.parameters():
        prm.grad = torch.ones_like(prm)
    opt.step()
    monkeypatch.setattr("%s._fused_ok" % type(opt).__module__, lambda *tensors: True)
    monkeypatch.setattr(pkg.norm_dist_cpp, "layer_ops", ops)
    for step in (3.0, torch.tensor(3.0), 3):
        for state in opt.state.values():
            state["step"] = step
        with pytest.raises(RuntimeError, match="CUDA"):   # as far as the look at the device, with every argument taken
            opt.step()


def test_tensors_past_the_native_range_are_left_to_torch(monkeypatch):
    """The native margins and attack step address 2^31 - 1 values; torch, which ran both before, takes more."""
    ops = mock.Mock()
    monkeypatch.setattr(pkg.norm_dist_cpp, "native_ops", lambda: ops)
    monkeypatch.setattr(pkg.AttackPGD, "_project", lambda self, x, centre=None: x)

    def tensor(rows, columns, dtype=torch.float32):
        t = mock.MagicMock(is_cuda=True, dtype=dtype, shape=(rows, columns))
        t.dim.return_value, t.numel.return_value, t.size.return_value = 2, rows * columns, rows
        for operation in ("__add__", "__sub__", "__rmul__"):
            getattr(t, operation).return_value = t
        return t

    for columns, native in ((1, True), (8, False)):
        t = tensor(2 ** 28, columns)
        pkg.BoundFinalIdentity()(t, t, t, tensor(2 ** 28, 1, torch.int64))
        pkg.AttackPGD(None, 0.1, 0.03, 3, 1.0, 0.0)._ascend(t, t, t)
        assert ops.margins.called == ops.pgd_step.called == native
        ops.reset_mock()


def test_attack_ranges_per_channel_are_left_to_torch(monkeypatch):
    """`down` and `up` may be anything that torch.as_tensor takes and that broadcasts; the native step takes numbers."""
    ops = mock.Mock()
    monkeypatch.setattr(pkg.norm_dist_cpp, "native_ops", lambda: ops)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))
    x, grad = torch.rand(2, 3, 4, 4), torch.randn(2, 3, 4, 4)
    low = np.array([0.1, 0.2, 0.3], dtype=np.float32).reshape(3, 1, 1)
    for down, up in ((low, 1.0), (0.0, low + 0.5), (low.tolist(), (low + 0.5).tolist())):
        got = pkg.AttackPGD(None, 0.1, 0.03, 1, up, down)._ascend(x, grad, x)
        want = torch.minimum(torch.maximum(x + 0.03 * grad.sign(), torch.as_tensor(down)), torch.as_tensor(up))
        assert not ops.pgd_step.called and torch.equal(got, want.float())
    pkg.AttackPGD(None, np.float32(0.1), 0.03, 1, 1, 0)._ascend(x, grad, x)
    assert ops.pgd_step.called


def test_an_attack_with_a_projection_of_its_own_uses_it(monkeypatch):
    """Replaced in a subclass or on the object: the native step knows the plain projection only."""
    ops = mock.Mock()
    monkeypatch.setattr(pkg.norm_dist_cpp, "native_ops", lambda: ops)
    monkeypatch.setattr(torch.Tensor, "is_cuda", property(lambda self: True))

    class Halved(pkg.AttackPGD):
        def _project(self, x, centre=None):
            return x / 2
    replaced = pkg.AttackPGD(None, 0.1, 0.03, 1, 1.0, 0.0)
    replaced._project = lambda x, centre=None: x / 2
    x, grad = torch.rand(2, 3, 4, 4), torch.randn(2, 3, 4, 4)
    for attack in (Halved(None, 0.1, 0.03, 1, 1.0, 0.0), replaced):
        assert torch.equal(attack._ascend(x, grad, x), (x + 0.03 * grad.sign()) / 2)
    assert not ops.pgd_step.called


def test_adamw_steps_what_comes_before_a_parameter_that_raises(monkeypatch):
    """The native loop takes its parameters together; those before a refused gradient have had their step all the same."""
    ops, net = mock.Mock(), torch.nn.Sequential(pkg.NormDist(6, 4, p=8.0), pkg.NormDist(4, 3, p=8.0))
    opt, params = pkg.AdamW(net), list(net.parameters())
    monkeypatch.setattr("%s._fused_ok" % type(opt).__module__, lambda *tensors: True)
    monkeypatch.setattr(pkg.norm_dist_cpp, "layer_ops", ops)
    for prm in params:
        prm.grad = torch.ones_like(prm)
    params[2].grad = params[2].grad.to_sparse()
    with pytest.raises(RuntimeError, match="sparse"):
        opt.step()
    (taken, _, _, _, hyper), _ = ops.adamw_step.call_args
    assert [id(t) for t in taken] == [id(t) for t in params[:2]]
    assert [h[-1] for h in hyper] == [opt.state[t]["step"] for t in params[:2]] == [1, 1]
    opt.param_groups[3]["lr"] = "none"             # the next one raises behind its count
    params[2].grad = torch.ones_like(params[2])
    with pytest.raises(ValueError):
        opt.step()
    (taken, *others, hyper), _ = ops.adamw_step.call_args
    assert len(taken) == len(hyper) == 3 and all(len(tensors) == 3 for tensors in others)
