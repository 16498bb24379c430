"""Batches whose reverse pass runs several groups of shots on each of the two
streams: a stream's table and slot list are overwritten by its next group, whose
shots start at the first step again, with captured chunks shared by groups of
one shape, and groups of different lengths.  Every shot equals the one migrated
alone.  tests/host_plan.cpp checks that these batches do have six groups or more
(lane_group_jobs there lists the same windows)."""
import numpy as np
import pytest

import gubingluo_amd as G

pytestmark = pytest.mark.gpu


def _job(nshot, ragged, **kw):
    nx, nz = 470, 300
    rng = np.random.default_rng(nshot)
    vp = np.sort(rng.uniform(1500.0, 3000.0, nz))[:, None] + rng.uniform(-20.0, 20.0, (nz, nx))
    d = dict(nshot=nshot, startshot=1, dshot=1, flag_layout=1, nx=nx, nz=nz, dx=10.0, dz=10.0, dt=1e-3, npml=32,
             fdom=25.0, spx0=1600.0, spz0=20.0, dspx=10.0, offsetmax=3000.0, direct=0.0, direct0=0.0)
    d.update(kw)
    om = None
    if ragged:                                             # windows of 61, 63 .. 299 columns, mixed
        om = np.array([10.0 * (60 + 2 * (37 * k % 120)) for k in range(nshot)], np.float32)
    return G.make_params(**d), vp.astype(np.float32), np.full((nz, nx), 2000.0, np.float32), om


@pytest.mark.parametrize("nshot,ragged,nt,kw", [
    (75, False, 64, dict(graph_chunk=25)),
    (75, False, 45, dict(graph_chunk=0)),
    (121, True, 55, dict(graph_chunk=20)),
    (121, True, 41, dict(graph_chunk=0)),
    # (snapshots start 4 / (fdom dt) = 160 steps in)
    (75, False, 231, dict(graph_chunk=50, store_fmt=G.STORE_F16, snap_every=20)),
    (75, False, 193, dict(graph_chunk=0, store_fmt=G.STORE_BF16, snap_every=10, snap_fmt=G.STORE_BF16)),
    (75, False, 48, dict(graph_chunk=16, ic_extra=True)),
])
def test_several_groups_a_stream(gpu_ctx, nshot, ragged, nt, kw):
    P, vp, rho, om = _job(nshot, ragged, nt=nt)
    print(f"[lane groups] {nshot} shots, ragged {ragged}, nt={nt} {kw}", flush=True)
    alone = dict(kw, graph_chunk=0)
    a = gpu_ctx.run(P, vp, rho, batch=0, want_shots=True, shot_offsetmax=om, **kw)
    b = gpu_ctx.run(P, vp, rho, batch=1, want_shots=True, shot_offsetmax=om, **alone)
    assert a.stats.batches == 1 and b.stats.batches == nshot
    for k in range(nshot):
        assert np.array_equal(a.shot_seis[k], b.shot_seis[k]), k
        assert np.array_equal(a.shot_g1[k], b.shot_g1[k]), k
        assert np.array_equal(a.shot_illum[k], b.shot_illum[k]), k
    assert np.abs(a.image1).max() > 0
    assert np.array_equal(a.image1, b.image1) and np.array_equal(a.image2s, b.image2s)
    for n in (a.ic or {}):
        assert np.array_equal(a.ic[n], b.ic[n]), n
    c = gpu_ctx.run(P, vp, rho, batch=0, shot_offsetmax=om, **kw)          # chunks captured by the first run
    assert np.array_equal(a.image1, c.image1) and np.array_equal(a.illum, c.illum)
