"""One transform's space domain on either side of the sizes from which backward calls
store it past the cache: 136 MiB, and 96 MiB for the x kernels with halved regions (192).
Class-split and split kernels, C2C and R2C, both precisions, against the FP64 oracle; the
forward call follows on the same field. Tolerances: 1e-12 (FP64) and 1e-5 (FP32), as the
same kernels have at smaller sizes."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.test_gpu_matrix import ellipsoid
from tests.test_gpu_parity import build, gpu_backward, gpu_forward
from tests.test_gpu_split_lengths import kernels_run
from tests.workloads import complex_values

pytestmark = pytest.mark.gpu

TOL = {"double": 1e-12, "float": 1e-5}


@pytest.mark.parametrize("plane,dims,r2c,precision", [
    (0, (192, 192, 240), False, "double"),  # 135 MiB
    (0, (192, 192, 252), False, "double"),  # 142 MiB
    (2, (192, 192, 168), False, "double"),  # 95 MiB
    (2, (192, 192, 180), False, "double"),  # 101 MiB
    (2, (210, 210, 200), False, "double"),  # 135 MiB
    (2, (210, 210, 210), False, "double"),  # 141 MiB
    (2, (256, 273, 256), True, "double"),   # 136.5 MiB, an odd number of rows
    (2, (256, 256, 280), False, "float"),   # 140 MiB
    (2, (256, 297, 480), True, "float"),    # 139 MiB
], ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else str(p))
def test_either_side(plane, dims, r2c, precision, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", str(plane))
    print(f"streaming limits: plane {plane} {dims} {r2c} {precision}", flush=True)
    t = ellipsoid(dims, 0.1, r2c)
    tr = build(dims, t, r2c, precision)
    o = orc.OraclePlan(r2c, dims, t)
    v = complex_values(0x5EED1F00 + len(t), len(t))
    want, got = o.backward(v), []
    ran = kernels_run(lambda: got.append(gpu_backward(tr, v, dims, r2c, precision)))
    assert ("k_xy_backward_fast" if plane == 0 else "k_xsplit_backward") in ran, ran
    assert orc.rel_l2(got[0], want) <= TOL[precision]
    assert orc.rel_l2(gpu_forward(tr, want, r2c, sp.SPFFT_FULL_SCALING, precision),
                      o.forward(want, True)) <= TOL[precision]
