"""16-row tiles shared by two workgroups (launches of up to 256 tiles): grid
heights that leave 1, 8, 9 or 16 rows to the last tile, so that its second
half is off the grid, holds one row or is whole, with the window's edges,
damping, strips, source and receivers in either half.  Every height computes
the same cells, so the results equal those of 32-row tiles bit for bit."""
import numpy as np
import pytest

import gubingluo_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz,npml,store", [(25, 20, G.STORE_F32), (32, 20, G.STORE_F32), (33, 20, G.STORE_F16),
                                           (40, 20, G.STORE_F32), (33, 16, G.STORE_F32), (70, 13, G.STORE_BF16)])
def test_halves_equal_whole_tiles(gpu_ctx, nz, npml, store):
    rng = np.random.default_rng(nz)
    nx = 150
    vp = (1900.0 + rng.uniform(0, 500, (nz, nx))).astype(np.float32)
    rho = (2000.0 + rng.uniform(-100, 100, (nz, nx))).astype(np.float32)
    P = G.make_params(nx=nx, nz=nz, nt=220, nshot=1, startshot=1, dshot=1, flag_layout=1, spx0=700.0, dspx=100.0,
                      offsetmax=600.0, npml=npml, dx=10.0, dz=10.0, dt=1e-3, fdom=20.0, spz0=20.0)
    a = gpu_ctx.run(P, vp, rho, tile_z=16, store_fmt=store, want_shots=True)
    b = gpu_ctx.run(P, vp, rho, tile_z=32, store_fmt=store, want_shots=True)
    print(f"[split] nz {nz} npml {npml} store {store}: {(nz + 2 * npml) % 16} rows in the last tile", flush=True)
    assert np.abs(a.image1).max() > 0
    assert np.array_equal(np.asarray(a.shot_seis[0]), np.asarray(b.shot_seis[0]))
    for k in ("image1", "image2s", "illum"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k
