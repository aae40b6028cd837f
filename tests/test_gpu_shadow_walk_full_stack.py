"""Rays through a dense cloud of triangles, whose pending nodes outgrow the
stack of the four-way walk: it walks a subtree in the binary records and goes
on with the stack. The flags equal the oracle's binary walk."""
import ctypes as C

import numpy as np
import pytest

import orc
from risltc_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("builder", [abi.BVH_SAH, abi.BVH_LBVH])
@pytest.mark.parametrize("n,size", [(30000, 0.4), (100000, 0.12)])
def test_dense_cloud(n, size, builder):
    import risltc_amd
    import torch
    rng = np.random.default_rng(n)
    tri = rng.uniform(-5, 5, (n, 1, 3)) + rng.normal(0, size, (n, 3, 3))
    mesh = synth.Mesh(tri, np.tile(np.array([0.0, 0.0, 1.0]), (n, 3, 1)), np.zeros((n, 3, 2)), np.zeros(n, int),
                      np.zeros(n, int))
    m = 20000
    o = rng.uniform(-7, 7, (m, 3))
    d = rng.normal(size=(m, 3))
    # short rays (most pass the cloud) and long ones
    tmax = np.where(np.arange(m) % 2 == 0, 20.0, rng.uniform(0.02, 0.4, m))
    rays = np.concatenate([o, np.full((m, 1), 1e-3), d, tmax[:, None]], 1).astype(np.float32)
    ctx = risltc_amd.Context(0)
    try:
        ctx.set_bvh_builder(builder)
        ctx.set_scene(mesh, [[0.5] * 6])
        hits = torch.full((m,), 7, dtype=torch.int32, device="cuda")
        ctx.trace_shadow_rays(torch.from_numpy(rays).cuda(), hits)
        torch.cuda.synchronize()
    finally:
        ctx.close()
    L, bvh = orc.lib(), orc.OrcBvh()
    dq = np.ascontiguousarray(mesh.dequantized(), np.float32)
    (L.orc_bvh_build_sah if builder == abi.BVH_SAH else L.orc_bvh_build)(C.byref(bvh), orc.ptr(dq, orc.f32p), n)
    o, d = np.ascontiguousarray(rays[:, 0:3]), np.ascontiguousarray(rays[:, 4:7])
    want = np.array([L.orc_bvh_any_hit(C.byref(bvh), orc.ptr(o[i], orc.f32p), orc.ptr(d[i], orc.f32p),
                                       float(rays[i, 3]), float(rays[i, 7]), None) for i in range(m)])
    L.orc_bvh_free(C.byref(bvh))
    got = hits.cpu().numpy()
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:10]
    assert 0.05 < want.mean() < 0.95
