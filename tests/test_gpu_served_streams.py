"""Served ticks whose forward and reverse steps run side by side on two
streams: shots of different lengths, so that forward and reverse launches,
phase changes, finished shots and reused slots (fewer slots than shots) meet
in every order, in fp32 and 16-bit strips.  Each request's images equal the
batch engine's own run of it, bit for bit."""
import numpy as np
import pytest

import gubingluo_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("store,slots", [(G.STORE_F32, 3), (G.STORE_F16, 2), (G.STORE_BF16, 8)])
def test_mixed_phases_equal_engine(gpu_ctx, store, slots):
    rng = np.random.default_rng(11)
    nz, nx = 70, 180
    vp = np.full((nz, nx), 2000.0, np.float32)
    vp[nz // 2:] = 2500.0
    vp += rng.uniform(-50, 50, (nz, nx)).astype(np.float32)
    rho = np.full((nz, nx), 2100.0, np.float32)
    mid = gpu_ctx.model_create(vp, rho)
    try:
        ps = [G.make_params(nx=nx, nz=nz, nt=nt, nshot=n, startshot=1, dshot=1, flag_layout=1, spx0=300.0,
                            dspx=200.0, offsetmax=off, npml=20, dx=10.0, dz=10.0, dt=1e-3, fdom=20.0, spz0=20.0)
              for nt, n, off in ((170, 3, 500.0), (290, 2, 900.0), (150, 4, 400.0), (201, 3, 700.0))]
        refs = [gpu_ctx.run(p, model=mid, store_fmt=store) for p in ps]
        with G.Server(gpu_ctx, max_slots=slots, store_fmt=store) as srv:
            ids = [srv.submit(mid, p) for p in ps]
            for i, (rid, p, ref) in enumerate(zip(ids, ps, refs)):
                i1, i2, il, lap, nrm, st = srv.wait(rid, p, timeout=60)
                print(f"[served streams] {store} {slots} slots: request {i}", flush=True)
                assert np.abs(ref.image1).max() > 0
                assert np.array_equal(i1, ref.image1) and np.array_equal(i2, ref.image2s)
                assert np.array_equal(il, ref.illum)
    finally:
        gpu_ctx.model_destroy(mid)
