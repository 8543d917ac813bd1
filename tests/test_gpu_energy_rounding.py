"""sparse_energy_batch of FP32 bands is the float64 sum of FP32 densities of fields
from the FFT kernels, whatever the tuner finds fastest for other calls: the
generic kernels' fields for lengths without fixed-length kernels, the split
stage's or the class-split kernels' for fixed ones. The reference is the same
loss as tensor expressions over those fields (which are equal bit for bit).

Tolerance: two FP64 sums of the same terms in different orders, each within
(number of terms) x 2^-53 of the sum of their absolute values."""
import numpy as np
import pytest

import spfft_amd as sp
from tests.test_gpu_matrix import ellipsoid
from tests.workloads import complex_values, uniform

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# the environment that the reference fields are made in
GENERIC, CLASS_SPLIT, SPLIT = (("SPFFT_AMD_GENERIC", "1"), ("SPFFT_AMD_PLANE", "0"),
                               ("SPFFT_AMD_PLANE", "2"))


@pytest.mark.parametrize("contiguous", [True, False], ids=["fused", "expression"])
@pytest.mark.parametrize("env,dims,bands", [
    (GENERIC, (20, 20, 20), 3), (GENERIC, (20, 20, 20), 1), (GENERIC, (31, 17, 24), 2),
    (GENERIC, (32, 32, 33), 2), (GENERIC, (67, 64, 64), 3), (SPLIT, (36, 48, 40), 3),
    (SPLIT, (60, 60, 45), 6), (CLASS_SPLIT, (64, 64, 64), 3), (CLASS_SPLIT, (32, 32, 36), 1),
], ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else str(p))
def test_energy_of_fft_fields(env, dims, bands, contiguous, monkeypatch):
    from spfft_amd.autograd import sparse_energy_batch
    nx, ny, nz = dims
    t = ellipsoid(dims, 0.3)
    print(f"energy rounding: {dims} x{bands} {env}", flush=True)

    def transforms():
        return [sp.TransformFloat(-1, sp.SPFFT_PU_GPU, sp.SPFFT_TRANS_C2C, *dims, len(t),
                                  sp.SPFFT_INDEX_TRIPLETS, t) for _ in range(bands)]

    c = np.stack([complex_values(0x5EED1600 + b, len(t)) for b in range(bands)])
    C = torch.from_numpy(c).to("cuda", torch.complex64)
    V = torch.from_numpy(uniform(0x5EED1620, nx * ny * nz).reshape(nz, ny, nx)).to(
        "cuda", torch.float32)
    if not contiguous:
        V = V.repeat_interleave(2, dim=2)[:, :, ::2]
    psi = torch.empty((bands, nz, ny, nx), dtype=torch.complex64, device="cuda")
    with monkeypatch.context() as m:
        m.setenv(*env)
        sp.multi_transform_backward(transforms(), list(C), list(psi))
    torch.cuda.synchronize()
    terms = V.to(torch.float64) * (psi.real ** 2 + psi.imag ** 2).to(torch.float64)
    want, bound = float(terms.sum()), terms.numel() * 2.0 ** -53 * float(terms.abs().sum())
    for plane in (None, "3"):
        with monkeypatch.context() as m:
            if plane:
                m.setenv("SPFFT_AMD_PLANE", plane)
            elif env == CLASS_SPLIT and bands > 1:
                m.setenv(*env)  # several FFT families serve the batch
            got = sparse_energy_batch(C, V, transforms(), dims)
        assert got.dtype == torch.float64
        assert abs(float(got) - want) <= bound, (plane, float(got), want)
