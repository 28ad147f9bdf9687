"""Behind the lists of outermost values (csrc/extremes_forward.hip) the kernels of the full walk are launched as well and leave at
once where the lists did the work: every kernel that a layer of any size takes, the one for a handful of rows included, which
narrow layers with a long reduction take at any batch."""
import pytest
import torch

from test_gpu_extremes import workspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1280, 416, 36864), (1200, 224, 30000), (512, 4096, 4096)])
@pytest.mark.parametrize("what", [0, 1, 2], ids=["positions", "values", "bounds"])
def test_the_full_walk_is_left_out(shape, what):
    from gpu_common import DEV, cpp, pkg, say
    B, CO, K = shape
    say("extremes gate", shape, what)
    assert workspace(B, CO, K, what) > 0
    g = torch.Generator(device=DEV).manual_seed(3)
    x, w = torch.rand(B, K, 1, device=DEV, generator=g), torch.randn(CO, K, device=DEV, generator=g) / K ** 0.5
    a, b = torch.empty(B, CO, 1, device=DEV), torch.empty(B, CO, 1, device=DEV)
    pos, up = torch.empty(B, CO, 1, device=DEV, dtype=torch.int32), x + 0.1

    def run():
        if what == 0:
            cpp.inf_dist_forward(x, w, a, pos, 1)
        elif what == 1:
            assert cpp.inf_dist_forward_values(x, w, a, 1)
        else:
            cpp.inf_dist_bound_forward(x, up, w, a, b, 1)

    def time_of(choice):
        """Shortest of seven, in ms."""
        pkg._lib.lib().ldist_set_extremes(choice)
        try:
            times = []
            for _ in range(8):
                start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                start.record()
                run()
                end.record()
                end.synchronize()
                times.append(start.elapsed_time(end))
            return min(times[1:])
        finally:
            pkg._lib.lib().ldist_set_extremes(-1)

    lists, full = time_of(-1), time_of(0)
    say(f"lists {lists:.3f} ms, full walk {full:.3f} ms")
    assert lists < 0.8 * full      # both together take more than the full walk alone
