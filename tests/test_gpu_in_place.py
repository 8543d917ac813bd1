"""Input and output in one buffer, against the FP64 oracle: values at the front, in
the middle and at the end of the field that a backward call writes, and in each
other's fields in a batch. Small sets of stick runs, whose values the matrix plane
kernel would read itself; and calls that would otherwise time the kernels.

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


# Shapes that no other test of the process tunes: the first call of each would be
# timed. Fixed lengths and a fixed length of z alone, spheres in stick runs (z
# kernels to choose from) and by shells.
TUNED = [(36, 40, 44), (40, 40, 40), (96, 96, 44), (22, 18, 36), (60, 35, 40)]


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("order", ["runs", "shells"])
@pytest.mark.parametrize("dims", TUNED, ids=lambda d: "x".join(map(str, d)))
def test_first_call_of_a_shape(dims, order, r2c, precision):
    print(f"in place, tuned: {dims} {order} {'R2C' if r2c else 'C2C'} {precision}", flush=True)
    t = ellipsoid(dims, 0.31 if order == "runs" else 0.27, r2c)
    if order == "shells":
        t = np.ascontiguousarray(t[np.argsort((t.astype(int) ** 2).sum(1), kind="stable")])
    n, o = int(np.prod(dims)) * (1 if r2c else 2), orc.OraclePlan(r2c, dims, t)
    v = complex_values(0x5EED1740 + n, len(t))
    s = o.backward(v)
    tr = build(dims, t, r2c, precision)
    buffer = torch.zeros(n, dtype=torch.float64 if precision == "double" else torch.float32,
                         device="cuda")
    buffer[:2 * len(t)] = reals(v, precision)
    tr.backward(buffer, buffer)
    tol = 1e-12 if precision == "double" else 1e-5
    assert orc.rel_l2(field_of(buffer, dims, r2c), s) <= tol
    tr.forward(buffer, buffer, sp.SPFFT_FULL_SCALING)
    got = buffer[:2 * len(t)].cpu().numpy().astype(np.float64).view(np.complex128)
    assert orc.rel_l2(got, o.forward(s, True)) <= tol


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("shift", [0, 1], ids=["own", "neighbours"])
@pytest.mark.parametrize("dims", [(36, 40, 48), (44, 44, 44), (21, 20, 36)],
                         ids=lambda d: "x".join(map(str, d)))
def test_first_batch_of_a_shape(dims, shift, precision):
    bands = 3
    print(f"in place batch, tuned: {dims} shift {shift} {precision}", flush=True)
    t = ellipsoid(dims, 0.31 + 0.02 * shift)
    n, o = 2 * int(np.prod(dims)), orc.OraclePlan(False, dims, t)
    trs = [build(dims, t, False, precision) for _ in range(bands)]
    fields = torch.zeros((bands, n), dtype=torch.float64 if precision == "double" else
                         torch.float32, device="cuda")
    vals = [complex_values(0x5EED1760 + b, len(t)) for b in range(bands)]
    values = [fields[(b + shift) % bands][:2 * len(t)] for b in range(bands)]
    for x, v in zip(values, vals):
        x.copy_(reals(v, precision))
    tol = 1e-12 if precision == "double" else 1e-5
    sp.multi_transform_backward(trs, values, list(fields))
    torch.cuda.synchronize()
    spaces = [o.backward(v) for v in vals]
    for b in range(bands):
        assert orc.rel_l2(field_of(fields[b], dims, False), spaces[b]) <= tol, b
    sp.multi_transform_forward(trs, list(fields), values, [sp.SPFFT_FULL_SCALING] * bands)
    torch.cuda.synchronize()
    for b in range(bands):
        got = values[b].cpu().numpy().astype(np.float64).view(np.complex128)
        assert orc.rel_l2(got, o.forward(spaces[b], True)) <= tol, b
