"""Input and output in one buffer, against the FP64 oracle: values at the front, in
the middle and at the end of the field that a backward call writes, and in each
other's fields in a batch. Small sets of stick runs, whose values the matrix plane
kernel would read itself.

Tolerances: those of the same kernels out of place, 1e-12 (FP64) and 1e-6 (FP32)."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.test_gpu_matrix import TOL, ellipsoid
from tests.test_gpu_parity import build, rdt
from tests.workloads import complex_values

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def field_of(buffer, dims, r2c):
    got = buffer.cpu().numpy().astype(np.float64)
    return (got if r2c else got.view(np.complex128)).reshape(dims[::-1])


def reals(v, precision):
    return torch.from_numpy(v.view(np.float64).astype(rdt(precision))).cuda()


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("dims", [(20, 20, 20), (24, 24, 24), (22, 18, 32)],
                         ids=lambda d: "x".join(map(str, d)))
def test_backward_of_small_sets(dims, r2c, precision, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", "3")
    print(f"in place: {dims} {'R2C' if r2c else 'C2C'} {precision}", flush=True)
    t = ellipsoid(dims, 0.3, r2c)
    n, o = int(np.prod(dims)) * (1 if r2c else 2), orc.OraclePlan(r2c, dims, t)
    v = complex_values(0x5EED1700 + n, len(t))
    for at in (0, (n // 4) // 2 * 2, n - 2 * len(t)):
        tr = build(dims, t, r2c, precision)
        buffer = torch.zeros(n, dtype=torch.float64 if precision == "double" else torch.float32,
                             device="cuda")
        buffer[at:at + 2 * len(t)] = reals(v, precision)
        tr.backward(buffer[at:], buffer)
        assert orc.rel_l2(field_of(buffer, dims, r2c), o.backward(v)) <= TOL[precision], at


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("shift", [0, 1], ids=["own", "neighbours"])
def test_backward_batches_of_small_sets(shift, precision, monkeypatch):
    """Band b's values in its own field, or in that of band b + 1."""
    monkeypatch.setenv("SPFFT_AMD_PLANE", "3")
    dims, bands = (20, 20, 20), 6
    print(f"in place batch: shift {shift} {precision}", flush=True)
    t = ellipsoid(dims, 0.3)
    n, o = 2 * int(np.prod(dims)), orc.OraclePlan(False, dims, t)
    trs = [build(dims, t, False, precision) for _ in range(bands)]
    dt = torch.float64 if precision == "double" else torch.float32
    fields = torch.zeros((bands, n), dtype=dt, device="cuda")
    vals = [complex_values(0x5EED1720 + b, len(t)) for b in range(bands)]
    ins = [fields[(b + shift) % bands][:2 * len(t)] for b in range(bands)]
    for x, v in zip(ins, vals):
        x.copy_(reals(v, precision))
    sp.multi_transform_backward(trs, ins, list(fields))
    torch.cuda.synchronize()
    for b in range(bands):
        assert orc.rel_l2(field_of(fields[b], dims, False), o.backward(vals[b])) <= TOL[precision], b
