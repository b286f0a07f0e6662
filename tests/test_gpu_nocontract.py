"""The parity build against the oracle, bit for bit.

The product library makes two rounding choices the oracle does not: the
compiler fuses a * b + c into one rounding (FMA contraction, as the
reference's --use_fast_math CUDA core also does), and stencil sums are
multiplied by a reciprocal of h^2 or h computed once, where the oracle (and
the reference's host core) divides.  On most cases the records move by ~1e-6
for it; the c1 case (two layers, order 4, a receiver on the interface)
amplifies it to ~4e-5 (test_oracle_acoustic2d.py::
test_fma_contraction_sensitivity_of_c1 shows the same shift in the oracle).

The parity build (sweep_amd/_lib/libswp_core_nocontract.so: the same sources
with -ffp-contract=off and SWP_EXACT_DIV) undoes both.  Loaded through
SWP_CORE_LIBRARY in a child process, so this process keeps the product
library, it must reproduce the oracle exactly -- any other difference in the
kernels' arithmetic (a term, an order of summation, a coefficient) shows as a
nonzero difference -- with two known exceptions, held to tighter bars:

* every record (2-D golden cases, 3-D and elastic random cases of orders
  2-10, both kernel families, full storage and boundary saving): exact;
* 2-D acoustic gradients: exact, both families, both modes;
* 3-D acoustic gradients: exact on the per-cell kernels.  The z-march
  adjoint forms the CPML term as (1 + b) * (v^2 dt^2 lambda), with
  v^2 dt^2 lambda taken from its plane queue, where the reference
  (acoustic3d/adjoint_split.cu:228-230) and the oracle form
  ((1 + b) * v^2 dt^2) * lambda: rel-L2 <= 1e-6 there (measured <= 5e-7);
* elastic gradients: exact in full storage.  With boundary saving the GPU
  images against velocities reconstructed by the reverse steps, the oracle
  against the stored forward ones (exact in exact arithmetic): the product
  bar, 1e-4 (measured <= 3.7e-5; the reference core's own boundary-saving
  fixtures pin this mode in test_gpu_elastic2d.py).
"""
from __future__ import annotations

import json
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]
TESTS = Path(__file__).resolve().parent
ORDERS = [2, 4, 6, 8, 10]
FAMILIES = ["auto", "zmarch"]
E_FIELDS = [(("vz",), ("vx", "vz")), (("vx",), ("vz", "sxx")), (("sxx",), ("szz",))]

_CHILD = r"""
import json, os, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
out_dir = sys.argv[2]
from conftest import GOLDEN
import test_gpu_acoustic2d as t2
import test_gpu_acoustic3d as t3
import test_gpu_elastic2d as te
import test_gpu_nocontract as tn
import torch
from sweep_amd import _core
dev = torch.device("cuda:0")

def family(fam):
    if fam == "auto":
        os.environ.pop("SWP_KERNELS", None)
    else:
        os.environ["SWP_KERNELS"] = fam

for name in t2.CASES:
    z = np.load(GOLDEN / f"acoustic2d_{name}.npz")
    for fam in tn.FAMILIES:
        family(fam)
        for mode in ("full", "bs"):
            print(f"[nocontract] acoustic2d {name} kernels={fam} mode={mode}", flush=True)
            np.savez(os.path.join(out_dir, f"a2d_{name}_{fam}_{mode}.npz"), **t2._run(z, mode, dev))
for order in tn.ORDERS:
    c = t3._random_case(order, seed=order)
    for fam in tn.FAMILIES:
        family(fam)
        for mode in ("full", "bs"):
            print(f"[nocontract] acoustic3d order={order} kernels={fam} mode={mode}", flush=True)
            r = t3._gpu_run(c["order"], c["shape"], c["dh"], c["dt"], c["abcn"], mode, c["vp"], c["wav"], c["src"],
                            c["rec"], c["res"], dev)
            np.savez(os.path.join(out_dir, f"a3d_{order}_{fam}_{mode}.npz"), **r)
family("auto")
for order in tn.ORDERS:
    for k, (st, rt) in enumerate(tn.E_FIELDS):
        c = te._random_case(order, seed=order)
        res = c["rng"].standard_normal((len(rt), c["B"], c["rec"].shape[1], c["nt"])).astype(np.float32)
        for mode in ("full", "bs"):
            print(f"[nocontract] elastic2d order={order} fields={k} mode={mode}", flush=True)
            r = te._gpu_run(order, c["shape"], c["dh"], c["dt"], c["abcn"], mode, c["models"], c["wav"], c["src"],
                            c["rec"], res, dev, list(st), list(rt))
            np.savez(os.path.join(out_dir, f"e2d_{order}_{k}_{mode}.npz"), res=res, **r)
print(json.dumps({"library": str(_core.library_path())}), flush=True)
"""


@pytest.fixture(scope="module")
def parity_runs(tmp_path_factory):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from sweep_amd.build import LIB_NOCONTRACT
    assert LIB_NOCONTRACT.exists(), "parity build missing: python -m sweep_amd.build --no-contract"
    out = tmp_path_factory.mktemp("nocontract")
    env = dict(os.environ, SWP_CORE_LIBRARY=str(LIB_NOCONTRACT), PYTHONPATH=str(ROOT))
    env.pop("SWP_KERNELS", None)
    print("[nocontract] child process on the parity build", flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", _CHILD, str(TESTS), str(out)], cwd=ROOT, env=env,
                       capture_output=True, text=True, timeout=400)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
    info = json.loads(r.stdout.strip().splitlines()[-1])
    assert Path(info["library"]) == LIB_NOCONTRACT.resolve()
    return out


def _compare(tag, got, ref, log):
    """Differing values and rel-L2 of each output; appended to log."""
    from conftest import rel_l2
    row = {}
    for k in ref:
        a, b = np.asarray(got[k], np.float32), np.asarray(ref[k], np.float32)
        assert a.shape == b.shape, (tag, k)
        row[k] = (int(np.count_nonzero(a != b)), rel_l2(a, b))
    print(f"[nocontract] {tag} (differing values, rel-L2) {row}", flush=True)
    log.append((tag, row))


def _check(log, exact):
    """Every output exact(tag, key) selects equal bit for bit; the others
    within the product bars (records 1e-5, gradients 1e-4)."""
    bad = []
    for tag, row in log:
        for k, (n, e) in row.items():
            if exact(tag, k):
                if n:
                    bad.append((tag, k, n, e))
            elif e > (1e-5 if k in ("rec", "obs", "pred") else 1e-4):
                bad.append((tag, k, n, e))
    assert not bad, bad


def test_acoustic2d_golden_cases_bit_exact(parity_runs):
    import test_gpu_acoustic2d as t2
    log = []
    for name in t2.CASES:
        for mode in ("full", "bs"):
            ref = t2._oracle(name, mode)
            for fam in FAMILIES:
                got = dict(np.load(parity_runs / f"a2d_{name}_{fam}_{mode}.npz"))
                _compare(f"acoustic2d {name} {fam} {mode}",
                         dict(obs=t2._raw(got["obs"]), pred=t2._raw(got["pred"]), grad_vp=got["grad_vp"],
                              grad_wavelet=got["grad_wavelet"]),
                         {k: ref[k] for k in ("obs", "pred", "grad_vp", "grad_wavelet")}, log)
    _check(log, lambda tag, k: True)


def test_acoustic3d_random_cases(parity_runs):
    import test_gpu_acoustic3d as t3
    log = []
    for order in ORDERS:
        c = t3._random_case(order, seed=order)
        for mode in ("full", "bs"):
            ref = t3._oracle_run(c, mode)
            for fam in FAMILIES:
                got = dict(np.load(parity_runs / f"a3d_{order}_{fam}_{mode}.npz"))
                _compare(f"acoustic3d order {order} {fam} {mode}", got, ref, log)
    zm_grad = lambda tag, k: " zmarch " in tag and k != "rec"
    _check(log, lambda tag, k: not zm_grad(tag, k))
    assert max(e for tag, row in log for k, (n, e) in row.items() if zm_grad(tag, k)) <= 1e-6


def test_elastic2d_random_cases(parity_runs):
    import test_gpu_elastic2d as te
    log = []
    for order in ORDERS:
        for k, (st, rt) in enumerate(E_FIELDS):
            c = te._random_case(order, seed=order)
            for mode in ("full", "bs"):
                got = dict(np.load(parity_runs / f"e2d_{order}_{k}_{mode}.npz"))
                ref = te._oracle_run(c, st, rt, got.pop("res"), bs=mode == "bs")
                _compare(f"elastic2d order {order} fields {k} {mode}", got, ref, log)
    _check(log, lambda tag, k: k == "rec" or tag.endswith(" full"))


def test_acoustic3d_roundings_of_the_large_sizes(tmp_path):
    """The forward kernel of 32M shot-cells and up differs from the smaller
    sizes' only in which products are fused: without contraction its records are
    the oracle's, bit for bit, too."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import test_gpu_acoustic3d as t3
    from sweep_amd.build import LIB_NOCONTRACT
    child = r"""
import os, sys
import numpy as np
sys.path.insert(0, sys.argv[1])
import test_gpu_acoustic3d as t3
import torch
for order in (2, 4, 6, 8):
    c = t3._random_case(order, seed=order)
    print(f"[nocontract] acoustic3d order={order} kernels=zmarch_big", flush=True)
    r = t3._gpu_run(c["order"], c["shape"], c["dh"], c["dt"], c["abcn"], "full", c["vp"], c["wav"], c["src"], c["rec"],
                    c["res"], torch.device("cuda:0"))
    np.savez(os.path.join(sys.argv[2], f"big_{order}.npz"), **r)
"""
    env = dict(os.environ, SWP_CORE_LIBRARY=str(LIB_NOCONTRACT), PYTHONPATH=str(ROOT), SWP_KERNELS="zmarch_big")
    r = subprocess.run([sys.executable, "-u", "-c", child, str(TESTS), str(tmp_path)], cwd=ROOT, env=env,
                       capture_output=True, text=True, timeout=400)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
    log = []
    for order in (2, 4, 6, 8):
        ref = t3._oracle_run(t3._random_case(order, seed=order), "full")
        _compare(f"acoustic3d order {order} zmarch_big full", dict(np.load(tmp_path / f"big_{order}.npz")), ref, log)
    _check(log, lambda tag, k: k == "rec")
