"""Rays from so far off that the error bound of the wide boxes exceeds whole
nodes: they meet a node's empty slots too, which must lead to one of its
triangles. The flags equal the oracle's binary walk."""
import ctypes as C

import numpy as np
import pytest

import orc
from risltc_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("builder", [abi.BVH_SAH, abi.BVH_LBVH])
@pytest.mark.parametrize("n", [2, 3, 7, 40])
def test_rays_from_far_off(n, builder):
    import risltc_amd
    import torch
    rng = np.random.default_rng(n)
    tri = (rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(0, 0.5, (n, 3, 3))) * 1e-5
    mesh = synth.Mesh(tri, np.tile(np.array([0.0, 0.0, 1.0]), (n, 3, 1)), np.zeros((n, 3, 2)), np.zeros(n, int),
                      np.zeros(n, int))
    ctx = risltc_amd.Context(0)
    ctx.set_bvh_builder(builder)
    ctx.set_scene(mesh, [[0.5] * 6])
    m = 1024
    o = rng.normal(size=(m, 3)).astype(np.float32)
    o *= (rng.uniform(10, 200, (m, 1)) / np.linalg.norm(o, axis=1, keepdims=True)).astype(np.float32)
    d = (rng.uniform(-2e-5, 2e-5, (m, 3)) - o).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.concatenate([o, np.zeros((m, 1)), d, np.full((m, 1), 1000.0)], 1).astype(np.float32)
    hits = torch.full((m,), 7, dtype=torch.int32, device="cuda")
    ctx.trace_shadow_rays(torch.from_numpy(rays).cuda(), hits)
    torch.cuda.synchronize()
    L, bvh = orc.lib(), orc.OrcBvh()
    dq = np.ascontiguousarray(mesh.dequantized(), np.float32)
    (L.orc_bvh_build_sah if builder == abi.BVH_SAH else L.orc_bvh_build)(C.byref(bvh), orc.ptr(dq, orc.f32p), n)
    o, d = np.ascontiguousarray(rays[:, 0:3]), np.ascontiguousarray(rays[:, 4:7])
    want = np.array([L.orc_bvh_any_hit(C.byref(bvh), orc.ptr(o[i], orc.f32p), orc.ptr(d[i], orc.f32p), 0.0, 1000.0,
                                       None) for i in range(m)])
    L.orc_bvh_free(C.byref(bvh))
    assert np.array_equal(hits.cpu().numpy(), want)
    ctx.close()
