"""Rays in a wall's plane whose direction leaves it by a denormal: its inverse is
infinite, the wall's own bounds let the ray pass (0 * inf), its parents' do
not. The flags equal the oracle's binary walk."""
import ctypes as C

import numpy as np
import pytest

import orc
from risltc_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("builder", [abi.BVH_SAH, abi.BVH_LBVH])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", [2, 3, 6, 40])
def test_denormal_direction(n, axis, builder):
    import risltc_amd
    import torch
    rng = np.random.default_rng(10 * n + axis)
    tri = rng.uniform(0, 20, (n, 3, 3))
    tri[:(n + 1) // 2, :, axis] = 0.0
    mesh = synth.Mesh(tri, np.tile(np.array([0.0, 0.0, 1.0]), (n, 3, 1)), np.zeros((n, 3, 2)), np.zeros(n, int),
                      np.zeros(n, int))
    # the quantisation puts the plane half a step off zero; here it is at zero
    mesh.dequantization_summand[:] = 0.0
    dq = np.ascontiguousarray(mesh.dequantized(), np.float32)
    assert np.all(dq.reshape(n, 3, 3)[:(n + 1) // 2, :, axis] == 0.0)
    m = 256
    wall = dq.reshape(n, 3, 3)[rng.integers(0, (n + 1) // 2, m)]
    o = np.einsum("ik,ika->ia", rng.dirichlet([1, 1, 1], m), wall).astype(np.float32)
    d = rng.normal(size=(m, 3)).astype(np.float32)
    d[:, axis] = rng.choice([-1, 1], m) * np.float32(2.5e-39)
    rays = np.concatenate([o, np.zeros((m, 1)), d, np.full((m, 1), 50.0)], 1).astype(np.float32)
    assert np.all(rays[:, 4 + axis] != 0.0)
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
    (L.orc_bvh_build_sah if builder == abi.BVH_SAH else L.orc_bvh_build)(C.byref(bvh), orc.ptr(dq, orc.f32p), n)
    o, d = np.ascontiguousarray(rays[:, 0:3]), np.ascontiguousarray(rays[:, 4:7])
    want = np.array([L.orc_bvh_any_hit(C.byref(bvh), orc.ptr(o[i], orc.f32p), orc.ptr(d[i], orc.f32p), 0.0, 50.0,
                                       None) for i in range(m)])
    L.orc_bvh_free(C.byref(bvh))
    assert np.array_equal(hits.cpu().numpy(), want)
