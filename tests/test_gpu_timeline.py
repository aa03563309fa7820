"""``ace_set_timeline``: only the fast forwards (softmax with class labels at
their channel counts), whose blocks the caller sized the buffer for, stamp
it."""

from __future__ import annotations

import pytest
import torch

from ace_kernels import ACEConfig, _lib, ace_loss
from ace_kernels.levels import ace_loss_levels
from gpu_helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("binning", ["hard", "soft"])
def test_only_fast_forwards_stamp(binning) -> None:
    lib = _lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(1)

    def case(channels, voxels, classes=True):
        x = torch.randn(1, channels, voxels, generator=gen, device="cuda")
        if classes:
            return x, torch.randint(0, channels, (1, 1, voxels), generator=gen, device="cuda")
        return x, (torch.rand(x.shape, generator=gen, device="cuda") < 0.3).float()

    labels = ACEConfig(binning=binning, num_bins=10, to_onehot_y=True)
    sigmoid = ACEConfig(binning=binning, num_bins=10, activation="sigmoid")
    raw = ACEConfig(binning=binning, num_bins=10, activation="none")
    voxels = 5000
    # room for every launch here, so that a stray stamp lands inside it
    buffer = torch.zeros(4096 * 8, dtype=torch.int64, device="cuda")
    others = {"wide labels": (case(5, voxels), labels), "wide targets": (case(4, voxels, False), sigmoid)}
    x, y = case(4, voxels, False)
    others["generic"] = ((torch.sigmoid(x), y), raw)
    xs, ys = zip(case(4, voxels), case(4, 640))
    x, y = case(4, voxels)
    say(f"timeline {binning}")
    try:
        _lib.check(lib.ace_set_timeline(buffer.data_ptr()), "ace_set_timeline")
        for name, ((a, b), cfg) in others.items():
            ace_loss(a, b, cfg)
            assert not bool(buffer.any()), name
        ace_loss_levels(list(xs), list(ys), labels)
        assert not bool(buffer.any()), "levels"
        ace_loss(x, y, labels)
        blocks = buffer.view(-1, 8)[:, 0].count_nonzero()
        assert 0 < int(blocks) <= -(-voxels // 256)
    finally:
        lib.ace_set_timeline(None)
