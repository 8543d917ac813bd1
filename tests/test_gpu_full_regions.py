"""FP64 batches on the split stage around 512 MiB of space domain, where the kernels of
192 and 256 change from halved to full LDS regions: which kernels run, and the results
against the FP64 oracle (first and last band). x and y of either kind (200 keeps its
halved regions), R2C with an odd number of planes and paired rows.

Tolerance: the operations are the same, 1e-12 as for every FP64 path."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.test_gpu_matrix import ellipsoid
from tests.test_gpu_parity import build
from tests.test_gpu_split_lengths import kernels_run
from tests.workloads import complex_values

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,r2c,count,x,y", [
    ((192, 192, 128), False, 7, "", ""),           # 504 MiB
    ((192, 192, 128), False, 8, "_full", "_full"),
    ((256, 200, 100), False, 7, "_full", ""),
    ((200, 256, 100), False, 7, "", "_full"),
    ((192, 256, 105), True, 14, "_full", "_full"),
    ((256, 192, 99), True, 14, "_full", "_full"),
], ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else str(p))
def test_large_batches(dims, r2c, count, x, y, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", "2")
    print(f"full regions: {count} x {dims} {'R2C' if r2c else 'C2C'}", flush=True)
    t = ellipsoid(dims, 0.12, r2c)
    n = int(np.prod(dims)) * (1 if r2c else 2)
    trs = [build(dims, t, r2c, "double") for _ in range(count)]
    vals = [complex_values(0x5EED1B00 + k, len(t)) for k in range(count)]
    ins = [torch.from_numpy(v.view(np.float64)).cuda() for v in vals]
    spaces = [torch.empty(n, dtype=torch.float64, device="cuda") for _ in trs]
    outs = [torch.empty(2 * len(t), dtype=torch.float64, device="cuda") for _ in trs]

    def run():
        sp.multi_transform_backward(trs, ins, spaces)
        sp.multi_transform_forward(trs, spaces, outs, [sp.SPFFT_FULL_SCALING] * count)
        torch.cuda.synchronize()

    ran = kernels_run(run)
    for way in ("backward", "forward"):
        assert {f"k_xsplit_{way}_batch{x}", f"k_ysplit_{way}_batch{y}"} <= ran, ran
    o = orc.OraclePlan(r2c, dims, t)
    for k in (0, count - 1):
        got = spaces[k].cpu().numpy()
        got = (got if r2c else got.view(np.complex128)).reshape(dims[::-1])
        assert orc.rel_l2(got, o.backward(vals[k])) <= 1e-12, k
        assert orc.rel_l2(outs[k].cpu().numpy().view(np.complex128), o.forward(got, True)) <= 1e-12
