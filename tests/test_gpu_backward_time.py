"""A gradient of 16-bit logits moves half the bytes of the same gradient of
float32 logits with the same arithmetic, and takes no longer."""

from __future__ import annotations

import statistics

import pytest
import torch

from ace_kernels import ACEConfig, _lib
from ace_kernels.impls import hip_mi355x as hip
from gpu_helpers import say

pytestmark = pytest.mark.gpu


def _backward_us(x, y, cfg) -> float:
    """Median kernel time of the backward, in turn with the forward."""
    lib, times = _lib.lib(), []
    go = torch.ones((), device="cuda")
    events = [tuple(torch.cuda.Event(enable_timing=True) for _ in range(2)) for _ in range(15)]
    for pair in events:
        for e in pair:
            e.record()  # creates the event
    for start, stop in events:
        pl = hip.make_plan(x, y, cfg)
        _, coef, d, jac, _, _ = hip.hip_forward(pl, cfg)
        lib.ace_set_launch_events(start.cuda_event, stop.cuda_event)
        hip.hip_backward(pl, coef, d, jac, go)
        lib.ace_set_launch_events(None, None)
    torch.cuda.synchronize()
    times = [start.elapsed_time(stop) * 1e3 for start, stop in events]
    return statistics.median(times[3:])


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("channels,bins,background", [(4, 20, True), (16, 20, True), (16, 50, False), (21, 20, True)])
def test_16_bit_gradient_takes_no_longer(channels, bins, background, binning) -> None:
    gen = torch.Generator(device="cuda").manual_seed(channels)
    voxels = 24_000_000 // channels
    x = torch.randn(1, channels, voxels, generator=gen, device="cuda") * 2.0
    y = torch.randint(0, channels, (1, 1, voxels), generator=gen, device="cuda")
    cfg = ACEConfig(binning=binning, num_bins=bins, to_onehot_y=True, include_background=background)
    say(f"backward time {binning} C={channels} K={bins} background={background}")
    full = _backward_us(x, y, cfg)
    half = {t: _backward_us(x.to(t), y, cfg) for t in (torch.bfloat16, torch.float16)}
    say(f"  float32 {full:.1f} us, " + ", ".join(f"{t} {v:.1f}" for t, v in half.items()))
    assert max(half.values()) <= 1.15 * full
