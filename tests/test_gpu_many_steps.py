"""Hard forwards whose blocks take more steps than 16 histogram copies can
count (above 7.8 M voxels at C <= 4)."""

from __future__ import annotations

import pytest
import torch

from ace_kernels import ACEConfig
from ace_kernels.common import bin_tables
from gpu_helpers import hip_stats, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels,voxels", [(4, 7_900_001), (4, 16_000_003), (2, 9_000_001), (3, 20_000_011)])
def test_many_steps_per_block(channels, voxels) -> None:
    """Hard forwards above 7.8 M voxels take 32 or 64 histogram copies: every
    voxel and label is counted once, and the bins are torch's but for
    probabilities within an ulp of an edge."""
    cfg = ACEConfig(binning="hard", num_bins=20, to_onehot_y=True)
    gen = torch.Generator(device="cuda").manual_seed(voxels)
    x = torch.randn(1, channels, voxels, generator=gen, device="cuda")
    y = torch.randint(0, channels, (1, 1, voxels), generator=gen, device="cuda")
    say(f"many steps C={channels} N={voxels}")
    st = hip_stats(x, y, cfg)[5]
    assert bool((st[0].sum(-1) == voxels).all())
    assert torch.equal(st[2][0].sum(-1), torch.bincount(y.flatten(), minlength=channels).double())
    p = torch.softmax(x, 1)
    edges = bin_tables(20, False, x.device)[0]
    for c in range(channels):
        counts = torch.bincount(torch.bucketize(p[0, c], edges), minlength=20).double()
        assert float((counts - st[0][0, c]).abs().sum()) <= 100
        assert abs(float(p[0, c].double().sum() - st[1][0, c].sum())) <= 2e-6 * voxels
