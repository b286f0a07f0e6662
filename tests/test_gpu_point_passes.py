"""Source and receiver passes that share a launch: the elastic fields of a
call, each alone, together, and listed twice (which keeps them apart)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sources,receivers", [
    (["vz"], ["vz", "vx", "sxx"]), (["sxx", "szz"], ["sxx", "vz"]), (["vz"], ["vz", "vz"]), (["vx", "vx"], ["vx"])])
def test_fields_of_a_call(sources, receivers):
    """Each channel of a record is what a call with that receiver field alone
    gives; a field listed twice as a source injects the wavelet twice."""
    from sweep_amd.equations import Elastic
    from sweep_amd.propagator import PropTorch
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(2)
    nt, shape = 70, (20, 26)
    vp = torch.tensor((2000 + 200 * rng.random(shape)).astype(np.float32), device=dev)
    models = [vp, vp / 1.8, 310.0 * vp ** 0.25]
    wav = (1e-3 * rng.standard_normal(nt)).astype(np.float32)
    src, rec = np.array([[8, 5], [15, 9]]), np.array([[[3, 2], [20, 7], [8, 5]], [[4, 4], [15, 9], [1, 1]]])

    def record(src_fields, rec_fields, w):
        solver = PropTorch(Elastic(spatial_order=4, device=dev), shape=shape, dh=5.0, dt=5e-4, device=dev, abcn=8,
                           source_type=src_fields, receiver_type=rec_fields)
        with torch.no_grad():
            return solver(w, src, rec, models=models)

    got = record(sources, receivers, wav)
    once = sorted(set(sources), key=sources.index)
    for k, field in enumerate(receivers):
        want = record(once, [field], wav * (len(sources) // len(once)))
        assert torch.allclose(got[..., k], want[..., 0], rtol=1e-5, atol=1e-6 * float(want.abs().max()))
