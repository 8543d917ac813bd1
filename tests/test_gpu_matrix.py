"""The matrix kernels (spfft_amd/csrc/dft_kernels.hip) against the FP64 oracle:
lengths without fixed-length kernels (below 32, primes, multiples of 17, ...)
on their own, and every plane they can serve with SPFFT_AMD_PLANE=3. The sizes
sit at the edges of their tiles: 16 lines by 16 output slots, where a slot
stands for two outputs of an odd length and four of an even one; lengths 4 m
(whose slot 0 also holds n / 4), 4 m + 2 and odd; one tile and several; planes
with few and many rows per workgroup; the longest length. C2C and R2C, both
precisions, spheres (stick runs), random columns (index tables), values in
random order, batches.

Tolerances: the sums have at most n / 2 + 1 terms in FP64, so their relative
error is below n * 2^-53 per stage, far inside the 1e-12 that the other FP64
paths are held to; FP32 results are rounded once per stage (3 * 2^-24, held to
1e-6 here, a tenth of the other FP32 paths' bound)."""
import numpy as np
import pytest

import spfft_amd as sp
from oracle import oracle as orc
from tests.test_gpu_parity import build, gpu_backward, gpu_forward, rdt
from tests.test_gpu_split_lengths import kernels_run
from tests.workloads import complex_values, random_index_set, sphere_triplets, uniform

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TOL = {"double": 1e-12, "float": 1e-6}
# no fixed-length kernels in any dimension
CUBIC = [1, 2, 3, 4, 5, 6, 7, 8, 15, 16, 17, 18, 20, 24, 30, 31, 33, 34, 58, 62, 65, 67, 97]
RAGGED = [(16, 17, 19), (31, 16, 22), (1, 30, 2), (29, 1, 64), (64, 62, 1), (127, 24, 33),
          (26, 128, 31), (251, 20, 16), (16, 254, 17), (18, 16, 253), (60, 31, 96), (34, 60, 128),
          (48, 36, 23)]
# planes that the fixed-length kernels serve too
FORCED = [(32, 32, 32), (36, 36, 36), (60, 60, 60), (64, 64, 40), (81, 75, 32), (96, 96, 32),
          (100, 100, 48), (128, 128, 32), (40, 48, 150), (256, 36, 32), (36, 256, 32)]


def check(dims, t, r2c, precision, seed):
    nx, ny, nz = dims
    print(f"matrix kernels: {dims} {'R2C' if r2c else 'C2C'} {precision}, {len(t)} values",
          flush=True)
    o = orc.OraclePlan(r2c, dims, t)
    tr = build(dims, t, r2c, precision)
    v = complex_values(seed, len(t))
    want = o.backward(v)
    assert orc.rel_l2(gpu_backward(tr, v, dims, r2c, precision), want) <= TOL[precision]
    s = uniform(seed + 1, nx * ny * nz).reshape(nz, ny, nx) if r2c else \
        complex_values(seed + 1, nx * ny * nz).reshape(nz, ny, nx)
    for scaling in (sp.SPFFT_NO_SCALING, sp.SPFFT_FULL_SCALING):
        f = gpu_forward(tr, s, r2c, scaling, precision)
        assert orc.rel_l2(f, o.forward(s, scaling == sp.SPFFT_FULL_SCALING)) <= TOL[precision]
    return tr


def ellipsoid(dims, fill, half=False):
    g = [np.arange(-((n - 1) // 2), (n - 1) // 2 + 1) for n in dims]
    x, y, z = np.meshgrid(*g, indexing="ij")
    keep = sum((c / max(1.0, fill * n)) ** 2 for c, n in zip((x, y, z), dims)) <= 1.0
    if half:
        keep &= (x > 0) | ((x == 0) & (y > 0)) | ((x == 0) & (y == 0) & (z >= 0))
    return np.ascontiguousarray(np.stack([x[keep], y[keep], z[keep]], axis=1).astype(np.int32))


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("dims", [(n, n, n) for n in CUBIC] + RAGGED,
                         ids=lambda d: "x".join(map(str, d)))
def test_free_lengths(dims, r2c, precision):
    seed = 0x5EED1000 + 7 * sum(dims)
    check(dims, ellipsoid(dims, 0.35, r2c), r2c, precision, seed)
    # every column, index and sign: dense random sets in storage order, shuffled
    t = random_index_set(seed + 2, dims, r2c, stick_fraction=0.8, fill_fraction=0.6)
    t = np.ascontiguousarray(t[np.argsort(uniform(seed + 3, len(t)), kind="stable")])
    if len(t):
        check(dims, t, r2c, precision, seed + 4)


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("dims", FORCED, ids=lambda d: "x".join(map(str, d)))
def test_planes_of_fixed_lengths(dims, r2c, precision, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", "3")
    seed = 0x5EED1100 + 7 * sum(dims)
    tr = check(dims, ellipsoid(dims, 0.3, r2c), r2c, precision, seed)
    v = complex_values(seed, tr.num_values)
    ran = kernels_run(lambda: gpu_backward(tr, v, dims, r2c, precision))
    assert "k_xy_backward_dft" in ran, ran
    t = random_index_set(seed + 2, dims, r2c, stick_fraction=0.3, fill_fraction=0.3, centered=True)
    check(dims, t, r2c, precision, seed + 4)


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("dims", [(20, 20, 20), (31, 33, 17), (60, 60, 48), (24, 97, 60)],
                         ids=lambda d: "x".join(map(str, d)))
def test_batches(dims, r2c, precision, monkeypatch):
    """Uneven sets (a sphere, a smaller one, a random one) in one call."""
    monkeypatch.setenv("SPFFT_AMD_PLANE", "3")
    seed = 0x5EED1200 + sum(dims)
    sets = [ellipsoid(dims, 0.35, r2c), ellipsoid(dims, 0.2, r2c),
            random_index_set(seed, dims, r2c, stick_fraction=0.4, fill_fraction=0.4)]
    n = int(np.prod(dims))
    rd = rdt(precision)
    dt = torch.float64 if precision == "double" else torch.float32
    trs = [build(dims, t, r2c, precision) for t in sets]
    vals = [complex_values(seed + k, len(t)) for k, t in enumerate(sets)]
    ins = [torch.from_numpy(v.view(np.float64).astype(rd)).cuda() for v in vals]
    spaces = [torch.empty(n * (1 if r2c else 2), dtype=dt, device="cuda") for _ in sets]
    outs = [torch.empty(2 * len(t), dtype=dt, device="cuda") for t in sets]
    print(f"matrix batch: {dims} {'R2C' if r2c else 'C2C'} {precision}", flush=True)
    sp.multi_transform_backward(trs, ins, spaces)
    sp.multi_transform_forward(trs, spaces, outs, [sp.SPFFT_FULL_SCALING] * len(trs))
    torch.cuda.synchronize()
    shape = (dims[2], dims[1], dims[0])
    for k, t in enumerate(sets):
        o = orc.OraclePlan(r2c, dims, t)
        got = spaces[k].cpu().numpy().astype(np.float64)
        got = got.reshape(shape) if r2c else got.view(np.complex128).reshape(shape)
        assert orc.rel_l2(got, o.backward(vals[k])) <= TOL[precision], k
        f = outs[k].cpu().numpy().astype(np.float64).view(np.complex128)
        assert orc.rel_l2(f, o.forward(got, True)) <= TOL[precision], k


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("dims", [(20, 20, 20), (21, 19, 23), (24, 24, 24), (16, 16, 2),
                                  (12, 12, 1), (8, 9, 64)], ids=lambda d: "x".join(map(str, d)))
def test_backward_from_values(dims, r2c, precision, monkeypatch):
    """Small sets of stick runs: the plane kernel sums the values over z itself,
    so no z kernel runs. Also runs that wrap, and whole sticks (z = n / 2 and a
    hermitian (0,0) stick with both halves given)."""
    monkeypatch.setenv("SPFFT_AMD_PLANE", "3")
    seed = 0x5EED1400 + sum(dims)
    whole = np.stack(np.meshgrid(*[np.arange(n // 2 + 1 if r2c and d == 0 else n)
                                   for d, n in enumerate(dims)], indexing="ij"), -1)
    whole = whole.reshape(-1, 3)
    whole = whole[(whole[:, 0] < 4) & (whole[:, 1] < 5)]
    for t in (ellipsoid(dims, 0.35, r2c), np.ascontiguousarray(whole.astype(np.int32))):
        assert len(t) <= 3000
        tr = check(dims, t, r2c, precision, seed)
        v = complex_values(seed, len(t))
        ran = kernels_run(lambda: gpu_backward(tr, v, dims, r2c, precision))
        assert ran == {"k_xy_backward_dft"}, ran
