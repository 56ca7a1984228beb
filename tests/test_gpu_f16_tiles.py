"""The matrix-core kernel of matmul_f16 (more than 8 columns, k % 16 == 0) at the edges of its tiles: each of
the four tile shapes (picked by the number of workgroups), ragged rows and columns, k below, at and past the
chunk of 256 values. Bar: the two-part activations are within 2^-22 of x and the sums of at most 8 + 8 partial
sums round at 2^-24 each: 2e-6 of each column's root mean square product sum, against float64."""
import numpy as np
import pytest

import kernelcore_amd as kc
from tests.test_gpu_f16 import case, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def runtime():
    kc.init()
    yield
    kc.synchronize()


@pytest.mark.parametrize("rows,k,ncols", [
    (8, 16, 9), (24, 240, 17), (40, 256, 16), (72, 272, 31), (520, 1040, 33),          # 16 x 16 tiles
    (1016, 512, 77), (1016, 768, 200), (2056, 272, 130), (4104, 528, 261),              # 32 x 16, 64 x 16, 64 x 32
    (8, 16, (1 << 20) + 20),                                                           # two launches
    (16384, 16, 10), (4104, 144, 261), (2056, 176, 1030), (16392, 272, 40),             # a 32 x 32 tile per wavefront
])
def test_matmul_f16_tiles(rows, k, ncols):
    print(f"matmul_f16 {rows} x {k} x {ncols}", flush=True)
    w, x = case(rows, k, ncols, rows + k + ncols)
    y = run(w, x, rows, k, ncols)
    w64, x64 = w.view(np.float16).astype(np.float64).reshape(rows, k), x.astype(np.float64).reshape(ncols, k)
    scale = np.sqrt((x64 ** 2) @ (w64 ** 2).T)
    assert (np.abs(y - x64 @ w64.T) <= 2e-6 * scale + 1e-30).all()
