"""The matrix kernels at their longest lines (257 to 320) as x, y and z, against the FP64
oracle: lengths without fixed-length kernels on their own, fixed ones with
SPFFT_AMD_PLANE=3, planes whose sticks no longer fit in LDS beside their rows (gathered),
dense sets of every index, and 321, which the generic kernels serve. The kernels that run
are named. Tolerances: as for shorter lines (the error of a sum grows with its terms:
161 x 2^-53 is far inside 1e-12)."""
import pytest

from tests.test_gpu_matrix import check, ellipsoid
from tests.test_gpu_parity import gpu_backward
from tests.test_gpu_split_lengths import kernels_run
from tests.workloads import complex_values, random_index_set

pytestmark = pytest.mark.gpu

FREE = [(319, 20, 16), (257, 16, 18), (16, 318, 17), (19, 311, 18), (18, 16, 319), (16, 17, 314),
        (317, 319, 3)]
FORCED = [(320, 36, 32), (36, 320, 32), (320, 320, 4), (288, 300, 5)]


@pytest.mark.parametrize("precision", ["double", "float"])
@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("dims", FREE + FORCED + [(321, 16, 16), (16, 16, 321)],
                         ids=lambda d: "x".join(map(str, d)))
def test_longest_lines(dims, r2c, precision, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", "3")
    seed = 0x5EED1D00 + 7 * sum(dims)
    tr = check(dims, ellipsoid(dims, 0.35, r2c), r2c, precision, seed)
    v = complex_values(seed, tr.num_values)
    ran = kernels_run(lambda: gpu_backward(tr, v, dims, r2c, precision))
    if max(dims) > 320:
        assert "k_z_backward" in ran and not any("_dft" in k for k in ran), ran
    else:
        assert "k_xy_backward_dft" in ran, ran
    t = random_index_set(seed + 2, dims, r2c, stick_fraction=0.5, fill_fraction=0.5)
    check(dims, t, r2c, precision, seed + 4)
