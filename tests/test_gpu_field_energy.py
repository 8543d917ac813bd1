"""The fused energy kernels of sparse_energy_batch against the same loss written
as torch expressions in float64: field sizes below, at and past a workgroup's
share (256 threads x 2 points, 64 workgroups x 4 points), one band and several,
both precisions, both recompute modes, an upstream factor on the loss, and a
potential that the kernels leave to tensor expressions (not contiguous).

Tolerances: energy and gradient are sums of one product per point, rounded once
per operation: 1e-12 in FP64; in FP32 the fields carry the transform's 1e-6."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.workloads import complex_values, uniform

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("contiguous", [True, False], ids=["fused", "expression"])
@pytest.mark.parametrize("recompute", [True, False])
@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("dims,bands", [((1, 2, 1), 1), ((8, 8, 8), 3), ((9, 3, 19), 2),
                                        ((41, 40, 40), 5)])
def test_energy_and_gradient(dims, bands, precision, recompute, contiguous):
    from spfft_amd.autograd import sparse_energy_batch
    nx, ny, nz = dims
    g = np.stack(np.meshgrid(*[np.arange(n) for n in dims], indexing="ij"), -1).reshape(-1, 3)
    t = np.ascontiguousarray(g[:: max(1, len(g) // 500)].astype(np.int32))
    kind = sp.Transform if precision == "double" else sp.TransformFloat
    ct, rt = ((torch.complex128, torch.float64) if precision == "double"
              else (torch.complex64, torch.float32))
    trs = [kind(-1, sp.SPFFT_PU_GPU, sp.SPFFT_TRANS_C2C, *dims, len(t), sp.SPFFT_INDEX_TRIPLETS, t)
           for _ in range(bands)]
    c = np.stack([complex_values(0x5EED1300 + b, len(t)) for b in range(bands)])
    v = uniform(0x5EED1320, nx * ny * nz).reshape(nz, ny, nx)
    C = torch.from_numpy(c).to("cuda", ct).requires_grad_(True)
    V = torch.from_numpy(v).to("cuda", rt)
    if not contiguous:
        V = V.repeat_interleave(2, dim=2)[:, :, ::2]
    print(f"energy: {dims} x{bands} {precision} recompute={recompute}", flush=True)
    (3.0 * sparse_energy_batch(C, V, trs, dims, recompute=recompute)).backward()
    energy = sparse_energy_batch(C, V, trs, dims, recompute=recompute)
    o = orc.OraclePlan(False, dims, t)
    want_e, want_g = 0.0, []
    for b in range(bands):
        psi = o.backward(c[b])
        want_e += np.sum(v * np.abs(psi) ** 2)
        want_g.append(3.0 * o.forward(2.0 * v * psi, False))
    tol = 1e-12 if precision == "double" else 1e-6
    assert energy.dtype == torch.float64
    assert abs(float(energy.detach()) - want_e) <= tol * np.sum(np.abs(v)) * np.sum(np.abs(c) ** 2)
    assert orc.rel_l2(C.grad.cpu().numpy().astype(np.complex128), np.stack(want_g)) <= tol
