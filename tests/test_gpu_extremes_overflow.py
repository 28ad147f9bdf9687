"""Lists of outermost values (csrc/extremes_forward.hip) of rows with more equal values at their outer end than a list has
places: constant rows (blank images) and saturated ones.  The search for a row's threshold t ends where no value should lie
beyond center +- t; with t = |v - center| the rounded center + t can still fall inside v, and then every copy of v counts as
beyond.  What does not fit the list must be covered by the row's bounds."""
import numpy as np
import pytest
import torch

import oracle
from helpers import gen

EPS = 8 / 255
LONGEST = 128      # places of the longest list, per chunk of at most 2560 inputs


def center_of(w):
    """extremes_sample_kernel's center in its order of additions: 1024 weights, a tree per wave, then the waves in turn."""
    rows, K = w.shape
    tid = np.arange(1024, dtype=np.int64)
    c = w.numpy()[tid * rows // 1024, tid * 61 % K].astype(np.float32).reshape(16, 64)
    for o in (32, 16, 8, 4, 2, 1):
        c = c + c[:, np.arange(64) ^ o]
    total = np.float32(0)
    for part in c[:, 0]:
        total = np.float32(total + part)
    return np.float32(total / np.float32(1024))


def beyond(v, center, boxes):
    """Whether all of a constant row's values count as beyond the threshold that they set themselves."""
    f = np.float32(2 if boxes else 1)
    key = f * np.float32(v)
    t = np.float32(np.abs(np.float32(key - f * center)) * np.float32(1 / f))
    return bool(key > f * np.float32(center + t) or key < f * np.float32(center - t))


def unsampled(rows):
    """Rows that the sample of 64 does not look at."""
    taken = {i * rows // 64 for i in range(64)}
    return [r for r in range(rows) if r not in taken]


def spread_rows(rows, K, seed, values, saturated):
    """N(0,1) rows of which the unsampled ones are constant, or in [0, 0.9) v with `saturated` of K equal to v."""
    m = torch.randn(rows, K, generator=gen(seed))
    for i, r in enumerate(unsampled(rows)):
        v = values[i // 2 % len(values)]
        if i % 2:
            m[r] = v
        else:
            m[r] = torch.rand(K, generator=gen(seed + r)) * (0.9 * v)
            m[r][torch.rand(K, generator=gen(seed - r)) < saturated] = v
    return m


def make(B, CO, K, side, offset, seed):
    """The constants are 1, -1, 1/2, grey values, and enough more that the rounding condition holds for several.  `offset` -0.7:
    the other operand's values lie a few units in the last place apart, so that a bound which is one unit off decides."""
    narrow = lambda rows: torch.randn(rows, K, generator=gen(seed + 7)) * (2.0 ** -23 if offset == -0.7 else K ** -0.5) + offset
    values = [1.0, -1.0, 0.5] + [u / 255 for u in (1, 37, 100, 128, 254)]
    more = [float(np.float32(0.3 + 0.013 * i)) for i in range(1, 200)]
    if side == "x":
        w = narrow(CO)
        values += [v for v in more if beyond(v, center_of(w), False)][:8]
        return spread_rows(B, K, seed, values, 0.15), w, values
    w = spread_rows(CO, K, seed, values, 0.15)        # the center is that of these rows, so it is known only now
    values += [v for v in more if beyond(v, center_of(w), False)][:8]
    for i, r in enumerate(unsampled(CO)):             # the sampled weights, and with them the center, must stay as they are
        used = {int(t) * CO // 1024 for t in range(1024)}
        if r not in used and i % 2:
            w[r] = values[i // 2 % len(values)]
    return narrow(B), w, values


# CO above 1024 on the weights' side: the center is the mean of 1024 weights, every row's below that
CASES = [("x", 200, 96, 5120, -0.7), ("x", 200, 96, 5120, -0.02), ("x", 200, 96, 5120, 0.02), ("x", 130, 300, 2560, 0.7), ("x", 200, 40, 1536, 0.0),
         ("w", 70, 1400, 2560, -0.02), ("w", 40, 1400, 5120, 0.3)]


@pytest.mark.parametrize("case", CASES)
def test_the_data_overflow_a_list(case):
    side, B, CO, K, offset = case
    x, w, values = make(B, CO, K, side, offset, seed=sum(case[1:4]))
    center = center_of(w)
    wide = x if side == "x" else w
    rows = [r for r in unsampled(wide.size(0)) if (wide[r] == wide[r, 0]).all() and beyond(float(wide[r, 0]), center, False)]
    assert len(rows) >= 3 and K > 2 * LONGEST
    assert side == "w" or any(beyond(float(wide[r, 0]), center, True) for r in rows)


@pytest.mark.gpu
@pytest.mark.parametrize("eps", [0.0, EPS])
@pytest.mark.parametrize("case", CASES)
def test_all_forms_match_the_oracle(case, eps):
    from gpu_common import DEV, cpp, gpu_bound_forward, gpu_inf_forward, pkg, say
    side, B, CO, K, offset = case
    say("extremes overflow", case, eps)
    x, w, _ = make(B, CO, K, side, offset, seed=sum(case[1:4]))
    x = x.unsqueeze(2).contiguous()
    lo, up = (x - eps).contiguous(), (x + eps).contiguous()
    pkg._lib.lib().ldist_set_extremes(1)
    try:
        out, pos = gpu_inf_forward(x, w, 1)
        only = torch.full((B, CO, 1), float("nan"), device=DEV)
        assert cpp.inf_dist_forward_values(x.to(DEV), w.to(DEV), only, 1)
        bounds = gpu_bound_forward(lo, up, w, 1)
    finally:
        pkg._lib.lib().ldist_set_extremes(-1)
    ev, ep = oracle.inf_dist_forward(x, w, 1)
    el, eu = oracle.inf_dist_bound_forward(lo, up, w, 1)
    pairs = {"values": (only.cpu(), ev), "values with positions": (out, ev), "positions": (pos, ep), "lower": (bounds[0], el),
             "upper": (bounds[1], eu)}
    assert {name: int((got != want).sum()) for name, (got, want) in pairs.items()} == dict.fromkeys(pairs, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("eps", [0.0, EPS])
def test_blank_images_in_a_batch_that_the_library_sends_this_way(eps):
    """1024 x 5120 -> 5120, against the full walk: ordinary rows, and a blank one for every grey value of a few."""
    from gpu_common import DEV, cpp, pkg, say
    B, CO, K = 1024, 5120, 5120
    say("extremes overflow, by the library", eps)
    g = torch.Generator(device=DEV).manual_seed(11)
    x, w = torch.randn(B, K, 1, device=DEV, generator=g), torch.randn(CO, K, device=DEV, generator=g) / K ** 0.5
    rows = unsampled(B)[::40]
    center = center_of(w.cpu())
    values = [v for v in [1.0, -1.0] + [float(np.float32(0.3 + 0.013 * i)) for i in range(1, 200)] if beyond(v, center, True)]
    assert len(rows) >= 16 and len(values) >= 1
    for i, r in enumerate(rows):
        x[r] = values[i % len(values)]
    lo, up = x - eps, x + eps

    def passes():
        a, b, c = (torch.full((B, CO, 1), float("nan"), device=DEV) for _ in range(3))
        only, pos = torch.full_like(a, float("nan")), torch.full((B, CO, 1), -7, device=DEV, dtype=torch.int32)
        cpp.inf_dist_bound_forward(lo, up, w, a, b, 1)
        cpp.inf_dist_forward(x, w, c, pos, 1)
        assert cpp.inf_dist_forward_values(x, w, only, 1)
        return a, b, c, pos, only

    got = passes()
    pkg._lib.lib().ldist_set_extremes(0)
    try:
        want = passes()
    finally:
        pkg._lib.lib().ldist_set_extremes(-1)
    assert [int((a != b).sum()) for a, b in zip(got, want)] == [0] * 5
