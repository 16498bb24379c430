"""A batch stepped in groups of shots on two streams: every shot equals the one
migrated alone, for batches of two groups, of several groups a stream (their
fields exceed what a group may hold) and of shots of different sizes, with
replayed chunks, plain launches and the autotuner's first steps."""
import numpy as np
import pytest

import gubingluo_amd as G

pytestmark = pytest.mark.gpu


def _job(nx, nz, nt, nshot, **kw):
    rng = np.random.default_rng(nx + nz)
    vp = np.sort(rng.uniform(1500.0, 3000.0, nz))[:, None] + np.zeros((nz, nx))
    d = dict(nshot=nshot, startshot=1, dshot=1, flag_layout=1, nx=nx, nz=nz, nt=nt, dx=10.0, dz=10.0, dt=1e-3, npml=32,
             fdom=25.0, spx0=300.0, spz0=20.0, dspx=10.0 * max(1, (nx - 60) // nshot), offsetmax=3000.0, direct=0.0,
             direct0=0.0)
    d.update(kw)
    return G.make_params(**d), vp.astype(np.float32), np.full((nz, nx), 2000.0, np.float32)


@pytest.mark.parametrize("nx,nz,nt,nshot,chunk,tz,ragged", [
    (300, 60, 120, 2, 10, 0, False),      # one shot a stream
    (300, 60, 61, 5, 0, 16, False),       # uneven groups, plain launches
    (400, 300, 64, 31, 25, 0, False),     # about 220 MB of fields: two groups a stream
    (400, 300, 40, 33, 0, 32, True),      # the same with windows of 60..350 columns
])
def test_groups_equal_single_shots(gpu_ctx, nx, nz, nt, nshot, chunk, tz, ragged):
    P, vp, rho = _job(nx, nz, nt, nshot)
    om = None
    if ragged:
        om = (np.linspace(60, 350, nshot)[::-1].round() * 10.0).astype(np.float32)
    print(f"[groups] {nshot} shots {nx}x{nz} nt={nt} chunk={chunk} tz={tz}", flush=True)
    kw = dict(want_shots=True, shot_offsetmax=om)
    a = gpu_ctx.run(P, vp, rho, batch=0, graph_chunk=chunk, tile_z=tz, **kw)
    b = gpu_ctx.run(P, vp, rho, batch=1, graph_chunk=0, tile_z=16, **kw)
    assert a.stats.batches == 1 and b.stats.batches == nshot
    for k in range(nshot):
        assert np.array_equal(a.shot_seis[k], b.shot_seis[k]), k
        assert np.array_equal(a.shot_g1[k], b.shot_g1[k]), k
        assert np.array_equal(a.shot_illum[k], b.shot_illum[k]), k
    assert np.array_equal(a.image1, b.image1) and np.array_equal(a.image2s, b.image2s)
    c = gpu_ctx.run(P, vp, rho, batch=0, graph_chunk=chunk, tile_z=tz, **kw)      # cached graphs and heights
    assert np.array_equal(a.image1, c.image1) and np.array_equal(a.illum, c.illum)
