"""The weight gradient at the edges of its tiles: strips of 64 / 128 columns and
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
