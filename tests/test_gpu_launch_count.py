"""The counters of launches count the launches that are made: a served tick's
steps, one more after a forward step of a 16-bit store; a timed pass's forward
steps, what follows them where something does, and its reverse steps."""
import numpy as np
import pytest

import gubingluo_amd as G

pytestmark = pytest.mark.gpu


def _job(nt):
    nx, nz = 150, 60
    vp = np.full((nz, nx), 2000.0, np.float32)
    vp[nz // 2:] = 2500.0
    P = G.make_params(nx=nx, nz=nz, nt=nt, nshot=1, startshot=1, dshot=1, flag_layout=2, spx0=700.0, spz0=20.0,
                      offsetmax=1500.0, npml=20, dx=10.0, dz=10.0, dt=1e-3, fdom=20.0)
    return P, vp, np.full((nz, nx), 2000.0, np.float32)


@pytest.mark.parametrize("store,forward", [(G.STORE_F32, 1), (G.STORE_F16, 2), (G.STORE_BF16, 2)])
def test_served_launches(gpu_ctx, store, forward):
    nt = 83
    P, vp, rho = _job(nt)
    mid = gpu_ctx.model_create(vp, rho)
    try:
        with G.Server(gpu_ctx, max_slots=2, store_fmt=store) as srv:
            print(f"[launches] served, store {store}", flush=True)
            srv.wait(srv.submit(mid, P), P, timeout=60)
            q = srv.query()
            assert q.ticks == 2 * nt - 1                   # one shot: a forward or a reverse step a tick
            assert q.launches == forward * nt + (nt - 1)
    finally:
        gpu_ctx.model_destroy(mid)


# snapshots start 4 / (fdom dt) = 200 steps in: none is due in 83 steps
@pytest.mark.parametrize("store,snap,nt,follows", [(G.STORE_F32, 0, 83, False), (G.STORE_F32, 20, 83, False),
                                                   (G.STORE_F32, 20, 300, True), (G.STORE_F16, 0, 83, True)])
def test_timed_steps(gpu_ctx, store, snap, nt, follows):
    P, vp, rho = _job(nt)
    print(f"[launches] timed, store {store}, snapshots {snap}, nt={nt}", flush=True)
    r = gpu_ctx.run(P, vp, rho, profile=True, store_fmt=store, snap_every=snap)
    assert list(r.stats.kern_calls) == [nt, nt if follows else 0, nt - 1, 0]
    assert (r.stats.kern_ms[1] > 0) == follows
    assert r.stats.kern_ms[0] > 0 and r.stats.kern_ms[2] > 0 and r.stats.kern_ms[3] == 0
    ref = gpu_ctx.run(P, vp, rho, store_fmt=store, snap_every=snap)
    assert np.array_equal(r.image1, ref.image1) and np.array_equal(r.illum, ref.illum)
