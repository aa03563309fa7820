"""The wide kernels (any channel count, softmax or sigmoid, class labels or
per-channel targets) against the CPU reference, at the edges of their channel
variants and of their steps, with fractional targets, right edges, extreme
logits, and against the generic kernels, which take a call whose workspace
holds only their sums."""

from __future__ import annotations

import pytest
import torch

from ace_kernels import ACEConfig, _lib, ace_loss
from ace_kernels.impls import hip_mi355x as hip
from gpu_helpers import LOSS_ATOL, LOSS_RTOL, assert_grad_close, run, say, truth64
from oracle.reference import reference_ace

pytestmark = pytest.mark.gpu

# both ends of the channel variants (a variant's first count pads most)
CHANNELS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 13, 14, 15, 16, 17, 20, 21, 24, 25, 32, 33, 48, 49, 64]


def _check(x, y, cfg) -> None:
    loss, grad = run("hip_mi355x", x.cuda(), y.cuda(), cfg)
    leaf = x.clone().requires_grad_(True)
    ref = reference_ace(leaf, y, cfg)
    (ref_grad,) = torch.autograd.grad(ref.sum(), leaf)
    loss64, grad64 = truth64(x, y, cfg)
    # the float32 reference's own distance from the float64 result on top
    err = (ref.detach().double() - loss64).abs()
    assert bool(((loss.cpu().double() - loss64).abs() <= err + LOSS_RTOL * loss64.abs() + LOSS_ATOL).all())
    few = cfg.binning == "soft" and x[0, 0].numel() < 100 * cfg.num_bins
    assert_grad_close(grad, ref_grad, x, cfg, rtol=1e-3 if few else 1e-4, truth=grad64)


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("channels", CHANNELS)
def test_labels(binning, channels) -> None:
    """Softmax with labels (sigmoid with one channel), an odd row past one step."""
    gen = torch.Generator().manual_seed(channels)
    x = torch.randn(2, channels, 33, 31, generator=gen) * 2.0
    one = channels == 1
    y = torch.randint(0, max(channels, 2), (2, 1, 33, 31), generator=gen)
    cfg = ACEConfig(binning=binning, num_bins=10, to_onehot_y=not one, include_background=channels % 3 != 0,
                    activation="sigmoid" if one else "softmax", right=channels % 2 == 0)
    say(f"wide labels {binning} C={channels}")
    _check(x, y.float() if one else y, cfg)


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("activation", ["softmax", "sigmoid"])
@pytest.mark.parametrize("channels,fractional", [(1, True), (2, False), (3, True), (4, True), (5, False), (7, True),
                                                 (17, True), (33, False), (64, True)])
def test_targets(binning, activation, channels, fractional) -> None:
    """Per-channel targets, among them values between 0 and 1 (label
    smoothing), which take sums of their own."""
    if channels == 1 and activation == "softmax":
        pytest.skip("softmax over one channel is no activation")
    gen = torch.Generator().manual_seed(100 + channels)
    x = torch.randn(2, channels, 1301, generator=gen) * 2.0
    y = (torch.rand(2, channels, 1301, generator=gen) < 0.3).float()
    if fractional:
        mix = torch.rand(y.shape, generator=gen)
        y = torch.where(mix < 0.3, mix, y)
    cfg = ACEConfig(binning=binning, num_bins=12, activation=activation, include_background=channels % 2 == 1)
    say(f"wide targets {binning} {activation} C={channels} fractional={fractional}")
    _check(x, y, cfg)


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("voxels", [1, 2, 3, 255, 256, 257, 511, 512, 513, 515, 1025, 4097])
def test_steps(binning, voxels) -> None:
    """Rows that end inside the first step, at its edge, one past it."""
    gen = torch.Generator().manual_seed(voxels)
    x = torch.randn(1, 6, voxels, generator=gen)
    y = torch.randint(0, 6, (1, 1, voxels), generator=gen)
    cfg = ACEConfig(binning=binning, num_bins=3, to_onehot_y=True)
    say(f"wide steps {binning} N={voxels}")
    _check(x, y, cfg)


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("channels", [5, 9])
def test_extreme_logits(channels, binning) -> None:
    """Saturated voxels match the reference; voxels with infinite or NaN logits
    leave every other voxel's gradient as it is with ordinary logits of the same
    probabilities in their place (a NaN or minus infinity beside finite logits:
    probability 0; plus infinity: all equal), and the loss too."""
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(1, channels, 2000, generator=gen)
    x[0, :, ::7] *= 400.0
    y = torch.randint(0, channels, (1, 1, 2000), generator=gen)
    cfg = ACEConfig(binning=binning, num_bins=10, to_onehot_y=True)
    say(f"wide extreme {binning} C={channels}")
    _check(x, y, cfg)
    # 12 bins: 1 / 5 and 1 / 9 lie far from every edge and centre
    cfg = ACEConfig(binning=binning, num_bins=12, to_onehot_y=True)
    x[0, :, 5:8] = torch.randn(channels, 3, generator=gen)
    low = x.clone()
    x[0, 0, 5], x[0, 1, 6], x[0, 2, 7] = float("inf"), float("-inf"), float("nan")
    low[0, :, 5], low[0, 1, 6], low[0, 2, 7] = 0.25, -1000.0, -1000.0
    loss, grad = run("hip_mi355x", x.cuda(), y.cuda(), cfg)
    loss_low, grad_low = run("hip_mi355x", low.cuda(), y.cuda(), cfg)
    torch.testing.assert_close(loss, loss_low, rtol=1e-6, atol=0)
    # hard: coefficients are counts and signs; soft: d moves by the last bit of
    # the equal probabilities
    others = torch.ones(2000, dtype=torch.bool)
    others[5:8] = False
    got, want = grad[0, :, others], grad_low[0, :, others]
    if binning == "hard":
        assert torch.equal(got, want)
    else:
        torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-9)


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("dtype,channels,voxels", [
    (torch.float32, 5, 1_100_003), (torch.bfloat16, 7, 1_700_001), (torch.float16, 13, 800_005),
    (torch.bfloat16, 21, 600_001), (torch.float32, 15, 2_100_001)])
def test_many_steps(dtype, channels, voxels, binning) -> None:
    """Blocks of several steps (two tiles in rotation, a row's end after full
    steps), 16-bit logits, and (the last one, 273 MB of logits, labels and
    gradient) streaming stores: the gradient equals to the bit that of pieces whose blocks
    take one step, from the same coefficients, and the hard forward's sums are
    the pieces' sums."""
    gen = torch.Generator(device="cuda").manual_seed(voxels)
    x = (torch.randn(1, channels, voxels, generator=gen, device="cuda") * 2.0).to(dtype)
    y = torch.randint(0, channels, (1, 1, voxels), generator=gen, device="cuda")
    cfg = ACEConfig(binning=binning, num_bins=20, to_onehot_y=True)
    say(f"wide many steps {binning} {dtype} C={channels} N={voxels}")
    go = torch.ones((), device="cuda")
    pl = hip.make_plan(x, y, cfg)
    _, coef, d, jac, _, st = hip.hip_forward(pl, cfg, stats=True)
    grad = hip.hip_backward(pl, coef, d, jac, go)
    total, at = torch.zeros_like(st), 0
    while at < voxels:
        n = min(99_991, voxels - at)
        piece = hip.make_plan(x[:, :, at:at + n].contiguous(), y[:, :, at:at + n].contiguous(), cfg)
        total += hip.hip_forward(piece, cfg, stats=True)[5]
        assert torch.equal(hip.hip_backward(piece, coef, d, jac, go), grad[:, :, at:at + n]), at
        at += n
    if binning == "hard":
        assert torch.equal(total, st)


def _stats(x, y, cfg, ws_bytes):
    """W, P, G of one forward given ws_bytes of workspace."""
    pl = hip.make_plan(x, y, cfg)
    lib, dev = _lib.lib(), x.device
    b, cl, k = pl.B, pl.CL, pl.K
    ws = torch.zeros(ws_bytes, dtype=torch.uint8, device=dev)
    coef, jac, per = (torch.empty(n, dtype=torch.float32, device=dev) for n in (b * cl * k, b * cl, b * cl))
    d = torch.empty(2 * b * cl * k, dtype=torch.float32, device=dev)
    loss = torch.empty((), dtype=torch.float32, device=dev)
    st = torch.empty(3, b, cl, k, dtype=torch.float64, device=dev)
    rc = lib.ace_forward(x.data_ptr(), pl.dtype_code, pl.target.data_ptr(), pl.target_kind, b, pl.C, pl.N, k,
                         _lib.SOFT if pl.soft else _lib.HARD, pl.act, int(pl.include_bg), 1, _lib.RED_MEAN,
                         int(pl.right), 0.01, None,
                         pl.btab.data_ptr(), hip._ptr(pl.rtab), ws.data_ptr(), ws_bytes, coef.data_ptr(),
                         d.data_ptr(), jac.data_ptr(), per.data_ptr(), loss.data_ptr(), st.data_ptr(), hip._stream(dev))
    return rc, loss, st, ws


@pytest.mark.parametrize("binning", ["hard", "soft"])
@pytest.mark.parametrize("kind", ["labels", "onehot", "fractional"])
@pytest.mark.parametrize("channels", [2, 5, 7])
def test_nan_probabilities(channels, kind, binning) -> None:
    """A NaN logit under a sigmoid has a NaN probability, which counts as 0:
    loss, sums and every other voxel's gradient are those of a logit of minus
    infinity in its place, in the wide kernels and (soft, a workspace of the
    generic size) in the generic ones."""
    gen = torch.Generator().manual_seed(channels)
    x = (torch.randn(2, channels, 1301, generator=gen) * 2.0).cuda()
    y = torch.randint(0, channels, (2, 1, 1301), generator=gen)
    if kind != "labels":
        y = torch.zeros(2, channels, 1301).scatter_(1, y, 1.0)
    if kind == "fractional":
        y = y * 0.8 + 0.1
    y = y.cuda()
    bad = torch.zeros(x.shape, dtype=torch.bool, device="cuda")
    bad[0, 0, 5] = bad[0, 1, 700] = bad[1, channels - 1, 1300] = True
    nan, low = x.masked_fill(bad, float("nan")), x.masked_fill(bad, float("-inf"))
    cfg = ACEConfig(binning=binning, num_bins=12, activation="sigmoid", to_onehot_y=kind == "labels")
    say(f"wide NaN {binning} C={channels} {kind}")
    (loss, grad), (loss_low, grad_low) = (run("hip_mi355x", t, y, cfg) for t in (nan, low))
    assert torch.equal(loss, loss_low) and torch.equal(grad[~bad], grad_low[~bad])
    sizes = [1 << 20]
    if binning == "soft":
        sizes.append(_generic_soft_bytes(2, channels, 1301, 12, kind == "labels"))
    for ws_bytes in sizes:
        (rc, *got), (rc_low, *want) = (_stats(t, y, cfg, ws_bytes)[:3] for t in (nan, low))
        assert rc == rc_low == 0 and all(torch.equal(a, b) for a, b in zip(got, want)), ws_bytes


def _generic_soft_bytes(b, channels, voxels, bins, labels) -> int:
    """Workspace bytes that hold the generic soft sums and no moments."""
    full = _lib.lib().ace_workspace_bytes(b, channels, voxels, bins, _lib.SOFT, 0, 1, 0 if labels else 1)
    return full - b * (7 if labels else 8) * channels * bins * 8 + 256  # (sizes are multiples of 256)


@pytest.mark.parametrize("channels,labels,activation,bins,right", [
    (5, True, "softmax", 20, False), (5, True, "softmax", 20, True), (8, True, "softmax", 50, False),
    (3, False, "softmax", 7, False), (4, False, "sigmoid", 20, True), (1, False, "sigmoid", 33, False),
    (17, True, "softmax", 10, False), (6, False, "softmax", 100, False), (1, False, "sigmoid", 512, False)])
def test_same_sums_as_the_generic_kernels(channels, labels, activation, bins, right) -> None:
    """(At many bins both sides run the generic kernel, the faster one there.)
    A workspace too small for the moments (ten or eleven words per bin) but
    large enough for the generic sums (three) selects the generic kernel: both
    give the same W, P and G to the generic kernel's fixed point (2^-39 a term
    at this size), and both leave their workspace zero."""
    gen = torch.Generator().manual_seed(bins)
    x = (torch.randn(2, channels, 3001, generator=gen) * 2.0).cuda()
    if labels:
        y = torch.randint(0, channels, (2, 1, 3001), generator=gen).cuda()
    else:
        y = torch.rand(2, channels, 3001, generator=gen)
        y = torch.where(y < 0.5, (y < 0.2).float(), y).cuda()
    cfg = ACEConfig(binning="soft", num_bins=bins, activation=activation, to_onehot_y=labels, right=right)
    say(f"wide vs generic C={channels} labels={labels} {activation} K={bins} right={right}")
    full = _lib.lib().ace_workspace_bytes(2, channels, 3001, bins, _lib.SOFT, 0, 1, 0 if labels else 1)
    rc, loss, wide, ws = _stats(x, y, cfg, full)
    assert rc == 0 and not bool(ws.any())
    # the generic layout's size: counters and partials, then 3 C'K words a batch index
    small = full - 2 * 7 * channels * bins * 8
    rc, loss_g, generic, ws = _stats(x, y, cfg, small)
    assert rc == 0 and not bool(ws.any())
    torch.testing.assert_close(wide, generic, rtol=0, atol=3001 * 2.0 ** -39)
    torch.testing.assert_close(loss, loss_g, rtol=1e-6, atol=1e-7)
    rc, *_ = _stats(x, y, cfg, 256)
    assert rc == 3  # ACE_EWORKSPACE


@pytest.mark.parametrize("channels,labels,activation,bins,voxels", [
    (5, True, "softmax", 50, 1_600_003), (8, True, "softmax", 50, 2_000_001), (14, True, "softmax", 20, 300_007),
    (1, False, "sigmoid", 50, 4_000_001), (4, False, "sigmoid", 100, 4_000_003), (8, False, "softmax", 20, 1_000_003)])
def test_large_problems_match_the_generic_kernels(channels, labels, activation, bins, voxels) -> None:
    """As above where many blocks of several steps run and the wide kernel is
    the faster one: tiles in rotation, copies near their count's limit, and
    replicas of the final sums."""
    gen = torch.Generator(device="cuda").manual_seed(bins)
    x = torch.randn(1, channels, voxels, generator=gen, device="cuda") * 2.0
    if labels:
        y = torch.randint(0, channels, (1, 1, voxels), generator=gen, device="cuda")
    else:
        y = torch.rand(1, channels, voxels, generator=gen, device="cuda")
        y = torch.where(y < 0.5, (y < 0.2).float(), y)
    cfg = ACEConfig(binning="soft", num_bins=bins, activation=activation, to_onehot_y=labels)
    say(f"wide vs generic C={channels} labels={labels} {activation} K={bins} N={voxels}")
    full = _lib.lib().ace_workspace_bytes(1, channels, voxels, bins, _lib.SOFT, 0, 1, 0 if labels else 1)
    rc, loss, wide, ws = _stats(x, y, cfg, full)
    assert rc == 0 and not bool(ws.any())
    rc, loss_g, generic, ws = _stats(x, y, cfg, _generic_soft_bytes(1, channels, voxels, bins, labels))
    assert rc == 0 and not bool(ws.any())
    # the generic kernels round each of a voxel's terms to half a unit of their
    # fixed point: 2^-41, coarser for more than 2^19 voxels (soft_frac)
    unit = 2.0 ** -min(40, 60 - voxels.bit_length())
    assert not torch.equal(wide, generic)  # two kernels
    torch.testing.assert_close(wide, generic, rtol=0, atol=voxels * unit)
    torch.testing.assert_close(loss, loss_g, rtol=1e-6, atol=1e-7)


def test_noalloc_scratch_limit() -> None:
    """A problem whose generic sums fit ace_forward_noalloc's 1 MiB and whose
    moments do not: still accepted, with the sums of ace_forward."""
    b, c, n, k = 30, 8, 600, 150
    gen = torch.Generator().manual_seed(9)
    x = torch.randn(b, c, n, generator=gen).cuda()
    y = torch.randint(0, c, (b, 1, n), generator=gen).cuda()
    cfg = ACEConfig(binning="soft", num_bins=k, to_onehot_y=True)
    lib, dev = _lib.lib(), x.device
    assert lib.ace_workspace_bytes(b, c, n, k, _lib.SOFT, 0, 1, 0) > 1 << 20
    pl = hip.make_plan(x, y, cfg)
    outs = [torch.empty(m, dtype=torch.float32, device=dev) for m in (b * c * k, 2 * b * c * k, b * c, b * c, 1)]
    say("wide noalloc at the scratch limit")
    rc = lib.ace_forward_noalloc(x.data_ptr(), 0, pl.target.data_ptr(), 0, b, c, n, k, _lib.SOFT, pl.act, 1, 1,
                                 _lib.RED_MEAN, 0, 0.01, None, pl.btab.data_ptr(), pl.rtab.data_ptr(),
                                 *[o.data_ptr() for o in outs], None, hip._stream(dev))
    assert rc == 0
    loss = ace_loss(x, y, cfg, impl="hip_mi355x")
    torch.testing.assert_close(outs[4][0], loss, rtol=1e-6, atol=1e-7)
