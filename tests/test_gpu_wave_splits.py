"""The three forms of a step of 16-row tiles, chosen by the tiles of a launch:
two workgroups of 8 rows a tile (up to 256 tiles), 8 waves of 2 rows (up to
384), 4 waves of 4 rows.  One shot is one launch a step, so its window says
which form runs; each equals the step of 32-row tiles shot by shot, with every
boundary store, in plain launches and in replayed chunks."""
import numpy as np
import pytest

import gubingluo_amd as G

pytestmark = pytest.mark.gpu


def _launch_tiles(nx, nz, npml):
    """16-row tiles of a full-aperture window.  A launch pads them for the 8
    XCDs to 8 runs of at most a quarter more than an eighth of them each."""
    n = -(-(nx + 2 * npml) // 64) * -(-(nz + 2 * npml) // 16)
    per = -(-n // 8)
    return n, 8 * (per + per // 4)


@pytest.mark.parametrize("store", [G.STORE_F32, G.STORE_F16, G.STORE_BF16])
@pytest.mark.parametrize("nx,nz,lo,hi", [
    (400, 163, 1, 256),                   # two workgroups a tile
    (690, 331, 257, 384),                 # 8 waves of 2 rows
    (811, 423, 385, 1 << 30),             # 4 waves of 4 rows
])
def test_16_row_forms_equal_32_rows(gpu_ctx, nx, nz, lo, hi, store):
    npml = 20
    n, most = _launch_tiles(nx, nz, npml)
    assert lo <= n and most <= hi                          # (whatever the padding is)
    rng = np.random.default_rng(nx)
    vp = rng.uniform(1500.0, 3000.0, (nz, nx)).astype(np.float32)
    rho = rng.uniform(1000.0, 2500.0, (nz, nx)).astype(np.float32)
    P = G.make_params(nshot=2, startshot=1, dshot=1, flag_layout=2, nx=nx, nz=nz, nt=171, dx=10.0, dz=10.0, dt=1e-3,
                      npml=npml, fdom=25.0, spx0=10.0 * (nx // 2), spz0=20.0, dspx=330.0, offsetmax=10.0 * nx,
                      alp=0.004, direct=0.0, direct0=0.0)
    print(f"[wave splits] {n} tiles, store {store}", flush=True)
    kw = dict(batch=1, want_shots=True, store_fmt=store)
    a = gpu_ctx.run(P, vp, rho, tile_z=32, **kw)
    assert np.abs(a.image1).max() > 0
    for chunk in (0, 25):
        b = gpu_ctx.run(P, vp, rho, tile_z=16, graph_chunk=chunk, **kw)
        for k in range(2):
            assert np.array_equal(a.shot_seis[k], b.shot_seis[k]), (chunk, k)
            assert np.array_equal(a.shot_g1[k], b.shot_g1[k]), (chunk, k)
            assert np.array_equal(a.shot_illum[k], b.shot_illum[k]), (chunk, k)
        assert np.array_equal(a.image1, b.image1) and np.array_equal(a.image2s, b.image2s)
