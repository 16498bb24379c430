"""The layer smoother's fronts at the sizes where they change form: the ring in
LDS or in memory (about 40000 floats apart), layers of 64 and 65 cells (63 and
64 lines of a wave; with 64 the last lane reads the line beside itself), odd
widths (a padded row), the smallest windows (3 layers a side) and layers of 2
cells.  Sums, their order and the number of sweeps are the host restatement's,
so results are equal bit for bit; so are windows with zeros (a relative change
of 0/0 or x/0), whose test is the same comparison."""
import numpy as np
import pytest

from tests.test_gpu_smoothing import host_smooth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,nx,npml", [
    (6, 6, 2), (9, 11, 3), (30, 31, 10), (96, 96, 32), (97, 300, 32),     # few or no rows between the layers
    (320, 265, 32), (300, 285, 33),                                      # ring in LDS, odd widths
    (240, 320, 33), (250, 333, 33),                                      # about the LDS limit, both sides
    (9, 4096, 3), (4096, 9, 3),                                          # lines far longer than the front
    (200, 195, 64), (200, 210, 65), (612, 401, 65),                      # 63 and 64 lines
])
def test_front_forms(gpu_ctx, nz, nx, npml):
    rng = np.random.default_rng(nz * 7 + nx)
    w = rng.uniform(1500.0, 4500.0, (nz, nx)).astype(np.float32) ** 2
    print(f"[front] {nz}x{nx} npml {npml}", flush=True)
    assert np.array_equal(gpu_ctx.smooth(w, npml=npml), host_smooth(w, npml=npml))


@pytest.mark.parametrize("nz,nx,npml", [(60, 61, 10), (420, 401, 50)])
def test_zeros(gpu_ctx, nz, nx, npml):
    rng = np.random.default_rng(3)
    w = rng.uniform(0.0, 1.0, (nz, nx)).astype(np.float32)
    w[rng.random((nz, nx)) < 0.3] = 0.0
    w[:, nx // 2:] = 0.0
    print(f"[front zeros] {nz}x{nx}", flush=True)
    assert np.array_equal(gpu_ctx.smooth(w, npml=npml), host_smooth(w, npml=npml))
