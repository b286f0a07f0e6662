"""The U-Net kernels at the edges of their tiles.  Weight gradient: strips of 64 / 128 columns and
their remainders, image rows fewer than a segment, each pairing of 32- and
64-channel tiles, channel counts that leave a tile part empty.  Against the
gradient of a float64 convolution of the same bf16 values; only the float32
summation differs, bar 1e-5 relative L2 as for the other convolutions.
"""
from __future__ import annotations

import pytest
import torch

from sweep_amd import _core
from sweep_amd.unet import _call, _p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W,cin,cout,ks", [
    (1, 1, 1, 8, 8, 3), (1, 3, 63, 64, 64, 3), (2, 4, 65, 64, 32, 3), (1, 9, 64, 40, 64, 3), (1, 5, 129, 32, 96, 3),
    (3, 2, 128, 8, 128, 3), (1, 21, 127, 192, 72, 3), (1, 7, 66, 64, 64, 1), (2, 3, 131, 32, 8, 1), (1, 2, 5, 64, 8, 1),
    (1, 4, 60, 8, 64, 1)])
def test_wgrad_tile_edges(N, H, W, cin, cout, ks):
    print(f"[unet] wgrad N={N} H={H} W={W} cin={cin} cout={cout} ks={ks}", flush=True)
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(H * 1000 + W + cin)
    x = torch.randn((N, H, W, cin), generator=g).to(torch.bfloat16)
    d = torch.randn((N, H, W, cout), generator=g).to(torch.bfloat16)
    r = ks // 2
    xp = torch.nn.functional.pad(x.double(), (0, 0, r, r, r, r))
    want = torch.stack([torch.tensordot(d.double(), xp[:, t // ks:t // ks + H, t % ks:t % ks + W],
                                        dims=([0, 1, 2], [0, 1, 2])) for t in range(ks * ks)], dim=1)
    dw = torch.full((cout, ks * ks, cin), float("nan"), device=dev)
    db = torch.empty(cout, device=dev)
    n = int(_core.load().swp_nn_conv_wgrad_scratch(N, H, W, cin, cout, ks))
    scratch = torch.full((n,), float("nan"), device=dev)
    xg, dg = x.to(dev), d.to(dev)
    _call("swp_nn_conv_wgrad", _p(xg), N, H, W, cin, cin, _p(dg), cout, cout, ks, _p(dw), _p(db), _p(scratch))
    got = dw.double().cpu()
    assert float((got - want).norm() / want.norm()) <= 1e-5
    assert float((db.double().cpu() - d.double().sum((0, 1, 2))).norm() / d.double().norm()) <= 1e-5


@pytest.mark.parametrize("N,H,W,cin,cout,ks", [
    (1, 1, 1, 8, 8, 3), (2, 3, 63, 32, 33, 3), (1, 5, 65, 40, 20, 3), (1, 4, 64, 64, 16, 3), (1, 9, 66, 72, 65, 3),
    (1, 2, 130, 104, 32, 3), (1, 6, 20, 128, 17, 3), (1, 3, 70, 136, 32, 3), (1, 3, 65, 32, 8, 1), (1, 2, 40, 96, 64, 1)])
def test_conv_tile_edges(N, H, W, cin, cout, ks):
    """The convolution at the edges of its 64 x 4 tiles, of its channel-count
    kernels (32, 64, 96, 128, more) and of its output tiles (16, 32, 64)."""
    print(f"[unet] conv N={N} H={H} W={W} cin={cin} cout={cout} ks={ks}", flush=True)
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(H * 1000 + W + cin + cout)
    x = torch.randn((N, H, W, cin), generator=g).to(torch.bfloat16)
    w = (torch.randn((cout, ks * ks, cin), generator=g) / (cin * ks * ks) ** 0.5).to(torch.bfloat16)
    b = torch.randn(cout, generator=g)
    r = ks // 2
    xp = torch.nn.functional.pad(x.double(), (0, 0, r, r, r, r))
    want = b.double() + sum(xp[:, t // ks:t // ks + H, t % ks:t % ks + W] @ w[:, t].double().t() for t in range(ks * ks))
    xg, wg, bg = x.to(dev), w.to(dev).contiguous(), b.to(dev)
    for os in (cout, cout + 3):
        out = torch.full((N, H, W, os), 7.0, device=dev)
        _call("swp_nn_conv_fwd", _p(xg), N, H, W, cin, cin, _p(wg), cout, ks, _p(bg), 0, _p(out), os, 1)
        got = out[..., :cout].double().cpu()
        assert float((got - want).norm() / want.norm()) <= 1e-5
        assert bool(torch.all(out[..., cout:] == 7.0))


def test_elementwise_passes_without_groups_of_eight():
    """Channel counts that are no multiple of 8 keep the one-channel passes."""
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(3)
    N, H, W, C = 1, 4, 6, 12
    x = torch.randn((N, H, W, C), generator=g).to(torch.bfloat16)
    xg = x.to(dev)
    p = torch.empty((N, H // 2, W // 2, C), dtype=torch.bfloat16, device=dev)
    _call("swp_nn_pool2_fwd", _p(xg), C, N, H, W, C, _p(p), C)
    v = x.float()
    want = ((v[:, 0::2, 0::2] + v[:, 0::2, 1::2]) + (v[:, 1::2, 0::2] + v[:, 1::2, 1::2])) * 0.25
    assert torch.equal(p.cpu(), want.to(torch.bfloat16))
    u = torch.empty((N, H, W, C), dtype=torch.bfloat16, device=dev)
    _call("swp_nn_up2_fwd", _p(p), C, N, H // 2, W // 2, C, _p(u), C)
    assert torch.equal(u.cpu(), p.cpu().repeat_interleave(2, 1).repeat_interleave(2, 2))
    d = torch.randn((N, H, W, C), generator=g).to(torch.bfloat16)
    dg = d.to(dev)
    _call("swp_nn_relu_bwd", _p(dg), C, _p(xg), C, N * H * W, C)
    assert torch.equal(dg.cpu(), torch.where(v > 0, d, torch.zeros_like(d)))


def test_negative_counts_are_empty():
    """A negative pixel or image count is an empty range, also for views that
    the eight-channel passes take."""
    dev = torch.device("cuda:0")
    H, W, C = 4, 4, 16
    a = torch.randn((1, H, W, C), device=dev).to(torch.bfloat16)
    b = torch.randn((1, 2 * H, 2 * W, C), device=dev).to(torch.bfloat16)
    a0, b0 = a.clone(), b.clone()
    _call("swp_nn_relu_bwd", _p(a), C, _p(b), C, -H * W, C)
    _call("swp_nn_pool2_fwd", _p(b), C, -1, 2 * H, 2 * W, C, _p(a), C)
    _call("swp_nn_pool2_bwd_acc", _p(a), C, -1, 2 * H, 2 * W, C, _p(b), C)
    _call("swp_nn_up2_fwd", _p(a), C, -1, H, W, C, _p(b), C)
    _call("swp_nn_up2_bwd", _p(b), C, -1, H, W, C, _p(a), C)
    assert torch.equal(a, a0) and torch.equal(b, b0)


@pytest.mark.parametrize("N,H,W,cin,cout,ks", [
    (50, 2, 130, 72, 40, 3), (50, 3, 65, 192, 128, 3), (90, 1, 65, 256, 128, 1), (37, 2, 129, 64, 520, 1)])
def test_wgrad_several_strips_a_workgroup(N, H, W, cin, cout, ks):
    """More strips of images than workgroups: each takes several in turn, the
    last ones perhaps fewer."""
    test_wgrad_tile_edges(N, H, W, cin, cout, ks)
