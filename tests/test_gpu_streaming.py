"""Large space domains against the FP64 oracle: at the sizes from which the
plane kernels write them with streaming stores (one transform from 96 MiB, a
batch from 144 MiB) and read them with streaming loads (from 256 MiB), just
below the first of them, and past it with rows in pairs of which the last is
single (R2C, odd ny). Every plane family: 0 class-split, 1 whole plane
(batches), 2 split stage, 3 matrix kernels.

Tolerances: streaming changes no operation, so the results are held to the
bounds of the same kernels at smaller sizes, 1e-12 (FP64) and 1e-5 (FP32)."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.test_gpu_matrix import ellipsoid
from tests.test_gpu_parity import build, gpu_backward, gpu_forward, rdt
from tests.workloads import complex_values, uniform

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {"double": 1e-12, "float": 1e-5}
SINGLE = [
    (0, (128, 128, 384), False, "double"),  # 96 MiB
    (2, (128, 128, 384), False, "double"),
    (2, (192, 192, 170), False, "double"),  # 95.6 MiB: plain
    (0, (192, 192, 351), True, "double"),
    (2, (256, 195, 256), True, "double"),
    (0, (192, 192, 351), False, "float"),
    (2, (256, 192, 256), False, "float"),   # 96 MiB
    (2, (256, 256, 256), False, "double"),  # 256 MiB
    (3, (256, 256, 256), False, "double"),
    (2, (512, 257, 256), True, "double"),
]


@pytest.mark.parametrize("plane,dims,r2c,precision", SINGLE,
                         ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else str(p))
def test_one_transform(plane, dims, r2c, precision, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", str(plane))
    print(f"large space domain: plane {plane} {dims} {r2c} {precision}", flush=True)
    t = ellipsoid(dims, 0.1, r2c)
    tr = build(dims, t, r2c, precision)
    o = orc.OraclePlan(r2c, dims, t)
    v = complex_values(0x57AE0000 + len(t), len(t))
    got = gpu_backward(tr, v, dims, r2c, precision)
    assert orc.rel_l2(got, o.backward(v)) <= TOL[precision]
    s = uniform(0x57AE1000 + len(t), got.size).reshape(got.shape)
    s = s if r2c else s - 1j * s[::-1, :, ::-1]
    assert orc.rel_l2(gpu_forward(tr, s, r2c, sp.SPFFT_FULL_SCALING, precision),
                      o.forward(s, True)) <= TOL[precision]


@pytest.mark.parametrize("plane,dims,r2c,precision,count", [
    (0, (128, 128, 64), False, "double", 9),   # 144 MiB
    (1, (64, 64, 64), False, "double", 36),
    (2, (100, 90, 128), False, "double", 10),
    (0, (128, 128, 64), True, "double", 18),
    (2, (128, 99, 128), True, "float", 26),
    (2, (128, 128, 128), False, "double", 8),  # 256 MiB
    (2, (256, 129, 128), True, "double", 8),
    (3, (97, 126, 128), False, "double", 11),
], ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else str(p))
def test_batches(plane, dims, r2c, precision, count, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", str(plane))
    print(f"large batch: plane {plane} {count} x {dims} {r2c} {precision}", flush=True)
    t = ellipsoid(dims, 0.15, r2c)
    n = int(np.prod(dims)) * (1 if r2c else 2)
    dt = torch.float64 if precision == "double" else torch.float32
    trs = [build(dims, t, r2c, precision) for _ in range(count)]
    vals = [complex_values(0x57AE2000 + k, len(t)) for k in range(count)]
    ins = [torch.from_numpy(v.view(np.float64).astype(rdt(precision))).cuda() for v in vals]
    spaces = [torch.empty(n, dtype=dt, device="cuda") for _ in trs]
    outs = [torch.empty(2 * len(t), dtype=dt, device="cuda") for _ in trs]
    sp.multi_transform_backward(trs, ins, spaces)
    sp.multi_transform_forward(trs, spaces, outs, [sp.SPFFT_FULL_SCALING] * count)
    torch.cuda.synchronize()
    o = orc.OraclePlan(r2c, dims, t)
    for k in (0, count - 1):
        got = spaces[k].cpu().numpy().astype(np.float64)
        got = got if r2c else got.view(np.complex128)
        got = got.reshape(dims[::-1])
        assert orc.rel_l2(got, o.backward(vals[k])) <= TOL[precision], k
        f = outs[k].cpu().numpy().astype(np.float64).view(np.complex128)
        assert orc.rel_l2(f, o.forward(got, True)) <= TOL[precision], k
