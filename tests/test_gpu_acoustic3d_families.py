"""Which 3-D kernel family a call runs on by default, from 4M shot-cells up,
where the choice depends on the order and the shape, and that it changes the
results by rounding alone: the record keeps its bits, a gradient moves by a few
float32 roundings.

Gradient bar 1e-5 relative L2: a value is the sum over the 24 steps of products of
two fields, each of whose steps adds some 30 roundings of 6e-8; all of one sign
that is 24 x 30 x 6e-8 = 4e-5, at random a thirtieth of it.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu

ABCN = 50


def _memory(name):
    from sweep_amd.options import BoundarySaving, Ckpt, Full
    return {"full": Full(), "bs": BoundarySaving(), "bs_bf16": BoundarySaving(storage_dtype="bf16"),
            "binomial": Ckpt(mode="recursive", count=5)}[name]


def _run(order, shape, B, mode, nt=24):
    """Record, model gradient and launch census of a call with its sources in
    corners and receivers around them, so that nt steps carry the wave to the
    receivers, over the strips and into the layers of every axis."""
    from sweep_amd import _core
    from sweep_amd.equations import Acoustic3D
    from sweep_amd.propagator import PropTorch
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(order + sum(shape))
    nz, ny, nx = shape
    z = np.linspace(0.0, 1.0, nz)[:, None, None]
    vp = (1800.0 + 900.0 * z + 100.0 * rng.random(shape)).astype(np.float32)
    t = np.arange(nt) * 1e-3
    a = (np.pi * 40.0 * (t - 0.006)) ** 2
    wav = ((1 - 2 * a) * np.exp(-a)).astype(np.float32)
    src = np.array([[3, 2, 2], [nx - 4, ny - 3, nz - 3]])[:B]
    off = np.stack(np.meshgrid([-2, 0, 2], [-2, 0, 2], [-1, 0, 1], indexing="ij"), -1).reshape(-1, 3)
    rec = src[:, None, :] + off[None]
    res = rng.standard_normal((B, nt, rec.shape[1], 1)).astype(np.float32)
    solver = PropTorch(Acoustic3D(spatial_order=order, device=dev), shape=shape, dh=10.0, dt=1e-3, device=dev, abcn=ABCN,
                       memory=_memory(mode))
    m = torch.tensor(vp, device=dev, requires_grad=True)
    _core.census_enable(True)
    pred = solver(wav, src, rec, models=[m])
    (pred * torch.tensor(res, device=dev)).sum().backward()
    torch.cuda.synchronize()
    sites = set(_core.census())
    _core.census_enable(False)
    return pred.detach(), m.grad.cpu().numpy(), sites


# order, shape, shots, memory, forward on the z-march, adjoint on it
ROUTES = [
    (2, (60, 60, 60), 1, "bs", True, True),
    (2, (38, 40, 147), 1, "bs", False, True),
    (2, (97, 110, 131), 1, "bs", True, True),
    (2, (80, 80, 80), 1, "bs_bf16", False, False),
    (2, (160, 160, 160), 1, "binomial", False, True),
    (4, (42, 28, 147), 1, "bs", False, True),
    (4, (40, 36, 44), 2, "bs", True, True),
    (4, (83, 28, 85), 1, "bs", False, False),
    (4, (80, 80, 80), 1, "binomial", False, True),
    (6, (83, 28, 85), 1, "full", False, True),
    (8, (83, 28, 85), 1, "bs", False, True),
    (8, (80, 80, 80), 1, "bs_bf16", True, True),
    (8, (40, 37, 45), 1, "bs", False, False),
    (10, (60, 60, 60), 1, "bs", False, False),
]


@pytest.mark.parametrize("order,shape,B,mode,fwd,adj", ROUTES)
def test_default_route(order, shape, B, mode, fwd, adj, monkeypatch):
    monkeypatch.delenv("SWP_KERNELS", raising=False)
    print(f"[families] order={order} shape={shape} B={B} {mode}", flush=True)
    rec, grad, sites = _run(order, shape, B, mode)
    for step, march in (("fwd", fwd), ("adj", adj)):
        assert any(s.startswith(f"a3d.{step}3.") for s in sites) == march, (step, sites)
        assert (f"a3d.{step}_cell" in sites) == (not march), (step, sites)
    monkeypatch.setenv("SWP_KERNELS", "percell")
    rec_cell, grad_cell, sites = _run(order, shape, B, mode)
    assert not any("3." in s[4:] for s in sites), sites
    e = rel_l2(grad, grad_cell)
    print(f"[families] {sorted(sites)} grad {e:.2e}", flush=True)
    assert torch.equal(rec, rec_cell)
    assert e <= 1e-5


@pytest.mark.parametrize("order,shape,mode,recon", [
    (8, (97, 63, 45), "bs", "cell"), (4, (50, 81, 67), "bs", "cell"), (8, (97, 63, 45), "bs_bf16", "cell"),
    (8, (176, 176, 176), "bs", "zm")])
def test_default_reconstruction(order, shape, mode, recon, monkeypatch):
    """Forward and adjoint on the z-march with a reconstruction box on either
    side of its own border: against full storage (the float32 strips; bar as for
    the full grids) and against the per-cell kernels."""
    monkeypatch.delenv("SWP_KERNELS", raising=False)
    print(f"[families] order={order} shape={shape} {mode}", flush=True)
    rec, grad, sites = _run(order, shape, 1, mode)
    assert any(s.startswith("a3d.fwd3.") for s in sites) and any(s.startswith("a3d.adj3.") for s in sites), sites
    assert {s for s in sites if s.startswith("a3d.recon")} == {f"a3d.recon_{recon}"}
    if mode == "bs":
        rec_full, grad_full, _ = _run(order, shape, 1, "full")
        e = rel_l2(grad, grad_full)
        print(f"[families] boundary saving against full {e:.2e}", flush=True)
        assert torch.equal(rec, rec_full)
        assert e <= 1e-4
    monkeypatch.setenv("SWP_KERNELS", "percell")
    rec_cell, grad_cell, _ = _run(order, shape, 1, mode)
    assert torch.equal(rec, rec_cell)
    assert rel_l2(grad, grad_cell) <= 1e-5


@pytest.mark.parametrize("order", [2, 4, 6, 8])
@pytest.mark.parametrize("mode", ["full", "bs"])
def test_roundings_of_the_large_sizes_match_oracle(order, mode, monkeypatch):
    """The forward kernel of 32M shot-cells and up, run on a small grid: every
    region type, records and gradients against the oracle, and a record that
    differs from the smaller sizes' by rounding."""
    import test_gpu_zmarch_interior as zi
    from sweep_amd.equations import Acoustic3D
    dev = torch.device("cuda:0")
    c = zi._case3d(order, seed=80 + order, B=1, nt=100)
    out = {}
    for family in ("zmarch", "zmarch_big"):
        monkeypatch.setenv("SWP_KERNELS", family)
        out[family] = zi._run(Acoustic3D(spatial_order=order, device=dev), c["shape"], c["dh"], c["dt"], c["abcn"], mode,
                              c["vp"], c["wav"], c["src"], c["rec"], c["res"], dev)
    got = out["zmarch_big"]
    for r in zi.REGIONS:
        assert got["census"].get(f"a3d.fwd3.{r}", (0, 0))[1] > 0, got["census"]
    ref = zi._oracle3d(c, mode)
    errs = {k: rel_l2(got[k], ref[k]) for k in ("rec", "grad_vp", "grad_wavelet")}
    moved = rel_l2(got["rec"], out["zmarch"]["rec"])
    print(f"[families] large-size roundings order {order} {mode} {errs}, record moved {moved:.1e}", flush=True)
    assert errs["rec"] <= 1e-5
    assert errs["grad_vp"] <= 1e-4
    assert errs["grad_wavelet"] <= 1e-4
    assert 0 < moved <= 1e-5
