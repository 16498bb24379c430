"""The step kernels' column quads at the sizes where they can go wrong: window
widths that end anywhere in a tile and in a quad, absorbing layers that start
anywhere in a quad, partial last tile rows, every tile height (16-row tiles in
both wave splits), bit for bit against the kernel-order oracle.  The source is
wide, so that the grid, its ring and its layer are non-zero from the first
step on."""
import numpy as np
import pytest

import gubingluo_amd as G
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _model(nz, nx, seed):
    rng = np.random.default_rng(seed)
    vp = rng.uniform(1500.0, 3000.0, (nz, nx)).astype(np.float32)
    rho = rng.uniform(1000.0, 2500.0, (nz, nx)).astype(np.float32)
    return vp, rho


@pytest.mark.parametrize("tz", [16, 32, 64])
@pytest.mark.parametrize("npml,nx,nz", [(10, 44, 30), (11, 107, 46), (13, 102, 45), (14, 163, 71), (15, 98, 98),
                                        (32, 65, 33), (10, 300, 130)])
def test_quads_vs_oracle(gpu_ctx, npml, nx, nz, tz):
    vp, rho = _model(nz, nx, npml + nx)
    kw = dict(nshot=1, startshot=1, dshot=1, flag_layout=2, nx=nx, nz=nz, nt=161, dx=10.0, dz=10.0, dt=1e-3, npml=npml,
              fdom=25.0, spx0=10.0 * (nx // 2) + 10.0, spz0=20.0, offsetmax=10.0 * nx, alp=0.004,
              direct=0.0, direct0=0.0)
    P, Po = G.make_params(**kw), O.make_params(**kw)
    print(f"[quads] npml={npml} {nx}x{nz} tz={tz}", flush=True)
    o = O.run_shot(Po, 1, vp, rho, korder=True)
    for chunk in (0, 10):
        r = gpu_ctx.run(P, vp, rho, tile_z=tz, graph_chunk=chunk, want_shots=True)
        assert np.array_equal(r.shot_seis[0], o.seis)
        assert np.array_equal(r.shot_g1[0], o.g1)
        assert np.array_equal(r.shot_illum[0], o.illum)
    assert np.abs(o.g1).max() > 0                          # some of the record is past the mute


def test_16_row_wave_splits_agree(gpu_ctx):
    """one shot (8 waves of 2 rows) against a batch past the split's bound (4
    waves of 4 rows), shot by shot"""
    nx, nz = 203, 150
    vp, rho = _model(nz, nx, 5)
    kw = dict(nshot=9, startshot=1, dshot=1, flag_layout=2, nx=nx, nz=nz, nt=60, dx=10.0, dz=10.0, dt=1e-3, npml=22,
              fdom=25.0, spx0=300.0, spz0=20.0, dspx=150.0, offsetmax=10.0 * nx, direct=0.0, direct0=0.0)
    P = G.make_params(**kw)
    print("[quads] 16-row splits", flush=True)
    a = gpu_ctx.run(P, vp, rho, tile_z=16, batch=1, want_shots=True)
    b = gpu_ctx.run(P, vp, rho, tile_z=16, batch=9, want_shots=True)      # 13 x 4 tiles a shot: 468 in all
    assert np.array_equal(a.image1, b.image1) and np.array_equal(a.illum, b.illum)
    for k in range(9):
        assert np.array_equal(a.shot_seis[k], b.shot_seis[k]) and np.array_equal(a.shot_g1[k], b.shot_g1[k])
