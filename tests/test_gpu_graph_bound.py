"""More captured chunks than an engine keeps (128): jobs of one shot whose chunk
lengths all differ take two each; the ones given back are captured again, and
every image equals the one of plain launches."""
import numpy as np
import pytest

import gubingluo_amd as G

pytestmark = pytest.mark.gpu


def test_more_chunks_than_are_kept():
    nx, nz, nt = 110, 50, 90
    vp = np.full((nz, nx), 2000.0, np.float32)
    vp[nz // 2:] = 2500.0
    rho = np.full((nz, nx), 2000.0, np.float32)
    P = G.make_params(nx=nx, nz=nz, nt=nt, nshot=1, startshot=1, dshot=1, flag_layout=2, spx0=500.0, spz0=20.0,
                      offsetmax=1100.0, npml=16, dx=10.0, dz=10.0, dt=1e-3, fdom=25.0, direct=0.0, direct0=0.0)
    with G.Context(0) as ctx:
        mid = ctx.model_create(vp, rho)
        ref = ctx.run(P, model=mid, graph_chunk=0)
        assert np.abs(ref.image1).max() > 0
        for chunk in list(range(1, 81)) + [1, 2, 40, 79, 80]:
            if chunk % 20 == 1:
                print(f"[graph bound] chunk {chunk}", flush=True)
            r = ctx.run(P, model=mid, graph_chunk=chunk)
            assert np.array_equal(r.image1, ref.image1) and np.array_equal(r.illum, ref.illum), chunk
        ctx.model_destroy(mid)
