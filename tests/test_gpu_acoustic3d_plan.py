"""The one-launch plan of the 3-D z-march at the shapes where it can go wrong:
region types without tiles (no pad on some faces, an empty interior), rows and
columns that leave partial tiles, z segments of the smallest height with a
remainder, one shot and several.  Records and gradients (full storage) against
the oracle; the strips and the reconstruction run in test_gpu_acoustic3d.py.

Bars as for every 3-D case: records rel-L2 <= 1e-5, gradients rel-L2 <= 1e-4.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import rel_l2
from test_gpu_acoustic3d import _canon, _dev

pytestmark = pytest.mark.gpu

# (order, shape, abcn, B): the interior is empty below 2 M + 3 cells an axis
CASES = [
    (2, (9, 7, 70), 4, 1),
    (4, (21, 12, 66), 5, 2),
    (6, (33, 18, 9), 3, 1),
    (8, (8, 9, 11), 6, 2),
    (8, (41, 35, 67), 7, 1),
    (8, (20, 40, 130), 2, 3),
]


@pytest.mark.parametrize("order,shape,abcn,B", CASES)
def test_plan_matches_oracle(order, shape, abcn, B, monkeypatch):
    from oracle.oracle import A3DProblem
    from sweep_amd.equations import Acoustic3D
    from sweep_amd.options import Full
    from sweep_amd.propagator import PropTorch
    dev = _dev()
    monkeypatch.setenv("SWP_KERNELS", "zmarch")
    print(f"[plan3d] order={order} shape={shape} abcn={abcn} B={B}", flush=True)
    rng = np.random.default_rng(order + sum(shape))
    nz, ny, nx = shape
    nt, dt, dh = 60, 9e-4, 9.0
    vp = (2000.0 + 300.0 * rng.random(shape)).astype(np.float32)
    a = (np.pi * 25.0 * (np.arange(nt) * dt - 0.03)) ** 2
    wav = ((1 - 2 * a) * np.exp(-a)).astype(np.float32)
    src = np.stack([rng.integers(0, n, B) for n in (nx, ny, nz)], -1)
    rec = np.stack([np.stack([rng.permutation(nx)[:3], rng.integers(0, ny, 3), rng.integers(0, nz, 3)], -1)
                    for _ in range(B)])
    res = rng.standard_normal((B, 3, nt)).astype(np.float32)
    solver = PropTorch(Acoustic3D(spatial_order=order, device=dev), shape=shape, dh=dh, dt=dt, device=dev, abcn=abcn,
                       memory=Full())
    m = torch.tensor(vp, device=dev, requires_grad=True)
    pred = solver(wav, src, rec, models=[m])
    (pred * torch.tensor(_canon(res), device=dev)).sum().backward()
    P = A3DProblem(order, shape, dh, dt, nt, abcn=abcn, B=B)
    w = np.ascontiguousarray(np.broadcast_to(wav, (B, 1, nt)))
    out = P.gradient(0, P.pad_model(vp), w, P.shift(src[:, None, :]), P.shift(rec), res)
    e_rec = rel_l2(pred.detach().cpu().numpy()[..., 0].transpose(0, 2, 1), out["rec"])
    e_g = rel_l2(m.grad.cpu().numpy(), P.crop(out["grad_vp"]).sum(0))
    print(f"[plan3d] rec {e_rec:.2e} grad {e_g:.2e}", flush=True)
    assert e_rec <= 1e-5
    assert e_g <= 1e-4


@pytest.mark.parametrize("order", [2, 4, 6, 8])
def test_record_bits_do_not_depend_on_the_family(order, monkeypatch):
    """Below the border of its larger sizes the z-march fixes its roundings to
    the per-cell kernel's: the two families' records are the same bits."""
    from sweep_amd.equations import Acoustic3D
    from sweep_amd.propagator import PropTorch
    dev = _dev()
    shape, nt, B = (14, 19, 33), 80, 2
    rng = np.random.default_rng(order)
    vp = torch.tensor((2000.0 + 300.0 * rng.random(shape)).astype(np.float32), device=dev)
    a = (np.pi * 25.0 * (np.arange(nt) * 9e-4 - 0.03)) ** 2
    wav = ((1 - 2 * a) * np.exp(-a)).astype(np.float32)
    src = np.array([[5, 6, 2], [30, 17, 11]])
    rec = np.stack([np.stack(np.meshgrid(np.arange(33), np.arange(19), [1], indexing="ij"), -1).reshape(-1, 3)] * B)
    out = {}
    for family in ("percell", "zmarch"):
        monkeypatch.setenv("SWP_KERNELS", family)
        solver = PropTorch(Acoustic3D(spatial_order=order, device=dev), shape=shape, dh=9.0, dt=9e-4, device=dev, abcn=6)
        with torch.no_grad():
            out[family] = solver(wav, src, rec, models=[vp])
    assert torch.equal(out["percell"], out["zmarch"])


@pytest.mark.parametrize("tz,least", [(64, 8), (48, 12), (9, 9), (5, 5)])
def test_segments_are_not_halved_below_eight_planes(tz, least, monkeypatch):
    """A launch of few waves halves its segment height while 8 planes or more
    remain: it starts as many workgroups as with that height kept."""
    from sweep_amd import _core
    from sweep_amd.equations import Acoustic3D
    from sweep_amd.propagator import PropTorch
    dev = _dev()
    monkeypatch.setenv("SWP_KERNELS", "zmarch")
    vp = torch.full((40, 30, 70), 2000.0, device=dev)
    wav = np.ones(3, np.float32)

    def census(height, waves):
        monkeypatch.setenv("SWP_TZ3", str(height))
        monkeypatch.setenv("SWP_REGION_WAVES", str(waves))
        solver = PropTorch(Acoustic3D(spatial_order=4, device=dev), shape=vp.shape, dh=9.0, dt=9e-4, device=dev, abcn=8)
        m = vp.clone().requires_grad_(True)
        _core.census_enable(True)
        solver(wav, np.array([[5, 6, 2]]), np.array([[[8, 6, 2]]]), models=[m]).sum().backward()
        torch.cuda.synchronize()
        out = {k: v for k, v in _core.census().items() if "3." in k[4:] or k == "a3d.recon_zm"}
        _core.census_enable(False)
        return out

    got = census(tz, 1 << 30)
    assert len(got) > 2
    assert got == census(least, 1)
