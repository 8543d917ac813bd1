"""Real space domains of 256 MiB and more on the split stage: rows stored and loaded in
pairs with streaming accesses, the last one single (odd ny). Against the FP64 oracle, with
the kernels named. Tolerance: 1e-12, as for every FP64 path."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.test_gpu_matrix import ellipsoid
from tests.test_gpu_parity import build
from tests.test_gpu_split_lengths import kernels_run
from tests.workloads import complex_values, uniform

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,count", [((512, 273, 256), 1), ((256, 135, 128), 8)],
                         ids=["one", "batch"])
def test_paired_rows(dims, count, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", "2")
    n = int(np.prod(dims))
    assert 8 * n * count >= 256 << 20
    print(f"streamed rows: {count} x {dims}", flush=True)
    t = ellipsoid(dims, 0.1, True)
    trs = [build(dims, t, True, "double") for _ in range(count)]
    vals = [complex_values(0x5EED1C00 + k, len(t)) for k in range(count)]
    ins = [torch.from_numpy(v.view(np.float64)).cuda() for v in vals]
    spaces = [torch.empty(n, dtype=torch.float64, device="cuda") for _ in trs]
    outs = [torch.empty(2 * len(t), dtype=torch.float64, device="cuda") for _ in trs]

    def backward():
        if count == 1:
            trs[0].backward(ins[0], spaces[0])
        else:
            sp.multi_transform_backward(trs, ins, spaces)

    def forward():
        if count == 1:
            trs[0].forward(spaces[0], outs[0], sp.SPFFT_FULL_SCALING)
        else:
            sp.multi_transform_forward(trs, spaces, outs, [sp.SPFFT_FULL_SCALING] * count)

    o = orc.OraclePlan(True, dims, t)
    tail = "_batch" if count > 1 else ""
    assert f"k_xsplit_backward{tail}" in kernels_run(backward)
    for k in sorted({0, count - 1}):
        got = spaces[k].cpu().numpy().reshape(dims[::-1])
        assert orc.rel_l2(got, o.backward(vals[k])) <= 1e-12, k
        # every point of its own, the single last rows too
        s = uniform(0x5EED1C40 + k, n).reshape(dims[::-1])
        spaces[k].copy_(torch.from_numpy(s.ravel()))
    assert f"k_xsplit_forward{tail}" in kernels_run(forward)
    torch.cuda.synchronize()
    for k in sorted({0, count - 1}):
        s = uniform(0x5EED1C40 + k, n).reshape(dims[::-1])
        f = outs[k].cpu().numpy().view(np.complex128)
        assert orc.rel_l2(f, o.forward(s, True)) <= 1e-12, k
