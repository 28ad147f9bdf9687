"""Which kernel a call takes, where another could serve: timed against the other, with margins well beyond the spread of a run."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def us(f):
    """Shortest of several replays of twenty calls."""
    f()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(20):
            f()
    graph.replay()
    times = []
    for _ in range(7):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        graph.replay()
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end) * 50)
    return min(times)


def data(B, CO, K):
    from gpu_common import DEV
    g = torch.Generator(device=DEV).manual_seed(B + CO + K)
    return (torch.rand(B, K, 1, device=DEV, generator=g), torch.randn(CO, K, device=DEV, generator=g) / K ** 0.5,
            torch.empty(B, CO, 1, device=DEV))


@pytest.mark.parametrize("case", [(1, 2, 12000, 37.3), (2, 3, 5120, 37.3), (2, 4, 40000, 8.0), (2, 4, 40000, None), (2, 8, 40000, None),
                                  (1, 10, 5120, 37.3), (2, 16, 3072, None)])
def test_few_outputs(case):
    """A workgroup per row, which a fixed choice of tiles keeps, or a wave per output: not more than a sixth slower."""
    from gpu_common import DEV, cpp, say, set_tile
    B, CO, K, p = case
    x, w, out = data(B, CO, K)
    pos = torch.empty(B, CO, 1, device=DEV, dtype=torch.int32)
    call = (lambda: cpp.inf_dist_forward(x, w, out, pos, 1)) if p is None else (lambda: cpp.norm_dist_forward_values(x, w, out, 1, p))
    chosen = us(call)
    set_tile(0)
    try:
        row = us(call)
    finally:
        set_tile(-1)
    say("few rows, few outputs", case, f"chosen {chosen:.1f} us, a workgroup per row {row:.1f} us")
    assert chosen < 7 / 6 * row


@pytest.mark.parametrize("case", [(31, 110, 28, 176, 2), (44, 7, 16, 159, 1), (31, 20, 32, 52, 4), (33, 48, 15, 62, 2)])
def test_channels_shared_by_groups_of_lanes(case):
    """Images with positions: the shape that is chosen is not slower than a tile to a group of lanes."""
    from gpu_common import DEV, cpp, pkg, say
    B, C, H, CO, G = case
    g = torch.Generator(device=DEV).manual_seed(B + C)
    x, w = torch.rand(B, C, H, H, device=DEV, generator=g), torch.randn(CO, C // G * 9, device=DEV, generator=g)
    out, pos = torch.empty(B, CO, H * H, device=DEV), torch.empty(B, CO, H * H, device=DEV, dtype=torch.int32)
    call = lambda: cpp.inf_dist_conv_forward(x, w, out, pos, G, 3, 1, 1)
    chosen = us(call)
    pkg._lib.lib().ldist_set_conv_groups_override(1)
    try:
        alone = us(call)
    finally:
        pkg._lib.lib().ldist_set_conv_groups_override(0)
    say("groups of lanes", case, f"chosen {chosen:.1f} us, a tile to a group {alone:.1f} us")
    assert chosen < 1.1 * alone
