"""Meshes whose dequantisation makes coordinates too large for areas, infinite
or NaN: their hierarchies are built, and the shadow flags equal the oracle's
binary walk (a triangle of coordinates that are not finite is never hit)."""
import ctypes as C

import numpy as np
import pytest

import orc
from risltc_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("builder", [abi.BVH_SAH, abi.BVH_LBVH])
@pytest.mark.parametrize("n", [3, 24, 98, 768])
@pytest.mark.parametrize("factor,summand", [(1e11, -1e17), (1e20, -1e26), (1e30, -1e36), (1e33, 0.0), (np.inf, 0.0),
                                            (1.0, np.nan), (1.0, np.inf), (np.nan, 0.0)])
def test_extent(n, factor, summand, builder):
    import risltc_amd
    import torch
    rng = np.random.default_rng(n)
    tri = rng.uniform(-5, 5, (n, 1, 3)) + rng.normal(0, 1.5, (n, 3, 3))
    mesh = synth.Mesh(tri, np.tile(np.array([0.0, 0.0, 1.0]), (n, 3, 1)), np.zeros((n, 3, 2)), np.zeros(n, int),
                      np.zeros(n, int))
    mesh.dequantization_factor[:] = factor
    mesh.dequantization_summand[:] = summand
    ctx = risltc_amd.Context(0)
    try:
        ctx.set_bvh_builder(builder)
        ctx.set_scene(mesh, [[0.5] * 6])
        m = 700
        size = 1e17 if factor < 1e15 else 1.0
        o = (rng.normal(size=(m, 3)) * size).astype(np.float32)
        d = rng.normal(size=(m, 3)).astype(np.float32)
        rays = np.concatenate([o, np.zeros((m, 1)), d, np.full((m, 1), np.inf)], 1).astype(np.float32)
        hits = torch.full((m,), 7, dtype=torch.int32, device="cuda")
        ctx.trace_shadow_rays(torch.from_numpy(rays).cuda(), hits)
        torch.cuda.synchronize()
    finally:
        ctx.close()
    with np.errstate(all="ignore"):
        dq = np.ascontiguousarray(mesh.dequantized(), np.float32)
    want = np.zeros(m, np.int32)
    if np.isfinite(dq).all():
        L, bvh = orc.lib(), orc.OrcBvh()
        (L.orc_bvh_build_sah if builder == abi.BVH_SAH else L.orc_bvh_build)(C.byref(bvh), orc.ptr(dq, orc.f32p), n)
        o, d = np.ascontiguousarray(rays[:, 0:3]), np.ascontiguousarray(rays[:, 4:7])
        want = np.array([L.orc_bvh_any_hit(C.byref(bvh), orc.ptr(o[i], orc.f32p), orc.ptr(d[i], orc.f32p), 0.0,
                                           float("inf"), None) for i in range(m)])
        L.orc_bvh_free(C.byref(bvh))
    else:
        assert not np.isfinite(dq).all(axis=1).any()
    assert np.array_equal(hits.cpu().numpy(), want)
