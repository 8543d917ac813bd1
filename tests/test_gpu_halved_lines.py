"""The split stage's FP64 kernels whose lines exchange through halved LDS regions
(and their tiles in two parts), against the FP64 oracle: every such length up to
512 as x and as y, with whole waves (192, 256, 320, 384, 512) and spare lanes
(200, 216, 500), next to lengths with full regions (96, 128, 45), R2C with an
odd number of rows, column counts that do and do not fill a workgroup. The
operations are those of the full regions, held to the same 1e-12."""
import pytest

from tests.test_gpu_matrix import check, ellipsoid
from tests.test_gpu_split_lengths import kernels_run
from tests.test_gpu_parity import gpu_backward
from tests.workloads import complex_values, random_index_set

pytestmark = pytest.mark.gpu

PLANES = [(192, 200), (216, 192), (256, 216), (320, 256), (200, 320), (384, 45), (45, 384),
          (448, 128), (96, 448), (512, 500), (500, 512)]


@pytest.mark.parametrize("r2c", [False, True], ids=["c2c", "r2c"])
@pytest.mark.parametrize("nx,ny", PLANES)
def test_halved_lines(nx, ny, r2c, monkeypatch):
    monkeypatch.setenv("SPFFT_AMD_PLANE", "2")
    dims = (nx, ny, 32)
    seed = 0x5EED1500 + nx + 3 * ny
    tr = check(dims, ellipsoid(dims, 0.3, r2c), r2c, "double", seed)
    v = complex_values(seed, tr.num_values)
    ran = kernels_run(lambda: gpu_backward(tr, v, dims, r2c, "double"))
    assert "k_ysplit_backward" in ran and "k_xsplit_backward" in ran, ran
    t = random_index_set(seed + 2, dims, r2c, stick_fraction=0.1, fill_fraction=0.3, centered=True)
    check(dims, t, r2c, "double", seed + 4)
