"""Vector loads at any element: rows of odd length and tensors that start at
any element of their storage run the same vectorised kernels as aligned ones.

Edges covered: rows shorter than one vector, one voxel beside a step or block
boundary (1023 / 1025, 16385), and storage offsets of 1-3 elements, which put
16-byte logit vectors, 16-byte label pairs and gradient stores at element
alignment only.  The offset run must equal the aligned run bit for bit (same
launch, same arithmetic); the longer rows also equal the CPU reference at the
parity tolerances.
"""

from __future__ import annotations

import pytest
import torch

from ace_kernels import ACEConfig, ace_loss
from gpu_helpers import LOSS_ATOL, LOSS_RTOL, assert_grad_close, run, say, truth64
from oracle.reference import reference_ace

pytestmark = pytest.mark.gpu


def _at_offset(t: torch.Tensor, offset: int) -> torch.Tensor:
    """A contiguous copy of t that starts `offset` elements into its storage."""
    flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=t.device)
    out = flat[offset:].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("channels,onehot", [(2, False), (3, False), (4, False), (5, False), (16, False), (4, True)])
def test_any_element(binning, dtype, channels, onehot) -> None:
    config = ACEConfig(binning=binning, num_bins=10, to_onehot_y=not onehot)
    for voxels, offset in ((1, 1), (3, 2), (1023, 1), (1025, 3), (16385, 1)):
        gen = torch.Generator().manual_seed(voxels + channels)
        x = (torch.randn(2, channels, voxels, generator=gen) * 1.5).to(dtype)
        y = torch.randint(0, channels, (2, 1, voxels), generator=gen)
        if onehot:
            y = torch.zeros(2, channels, voxels).scatter_(1, y, 1.0)
        say(f"unaligned {binning} {dtype} C={channels} onehot={onehot} N={voxels} offset={offset}")
        loss, grad = run("hip_mi355x", x.cuda(), y.cuda(), config)
        xo, yo = _at_offset(x.cuda(), offset).requires_grad_(True), _at_offset(y.cuda(), offset)
        loss_o = ace_loss(xo, yo, config, impl="hip_mi355x")
        (grad_o,) = torch.autograd.grad(loss_o, xo)
        assert torch.equal(loss, loss_o.detach()) and torch.equal(grad, grad_o)
        if voxels < 1000:
            continue
        leaf = x.float().clone().requires_grad_(True)
        ref = reference_ace(leaf, y, config)
        torch.testing.assert_close(loss.cpu(), ref.detach(), rtol=LOSS_RTOL, atol=LOSS_ATOL)
        if dtype == torch.float32:
            (ref_grad,) = torch.autograd.grad(ref, leaf)
            _, truth = truth64(x, y, config)
            assert_grad_close(grad, ref_grad, x, config, truth=truth)
