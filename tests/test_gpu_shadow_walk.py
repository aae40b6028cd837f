"""The shadow walk over four-way nodes against the oracle's binary walk: the
same flag for every ray, on trees of one leaf and up, both builders, and the
rays at the limits of the wide boxes' error bound."""
import ctypes as C

import numpy as np
import pytest

import orc
from risltc_amd import abi, synth

pytestmark = pytest.mark.gpu


def soup(n, kind, rng):
    if kind == "pile":
        # overlapping right triangles: every box on a path is met, so the
        # pending nodes of a walk outgrow its stack
        base = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.2], [0.0, 1.0, 0.2]])
        tri = base[None] + rng.uniform(-1e-3, 1e-3, (n, 3, 3))
    else:
        tri = rng.uniform(-5, 5, (n, 1, 3)) + rng.normal(0, 0.8, (n, 3, 3))
        if kind == "flat":
            # walls parallel to the axes: boxes without extent
            a = rng.integers(0, 3, n)
            tri[np.arange(n), :, a] = tri[np.arange(n), :1, a]
    return synth.Mesh(tri, np.tile(np.array([0.0, 0.0, 1.0]), (n, 3, 1)), np.zeros((n, 3, 2)), np.zeros(n, int),
                      np.zeros(n, int))


def rays_for(rng, n):
    o = rng.uniform(-7, 7, (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    tmin, tmax = np.full(n, 1e-3, np.float32), rng.uniform(0.1, 20, n).astype(np.float32)
    k = np.arange(n) % 24
    for a in range(3):
        d[k == a, a] = 0.0                       # parallel to a plane
        d[k == 3 + a] = np.eye(3, dtype=np.float32)[a] * 2  # parallel to an axis
        d[k == 6 + a, a] = 1e-6                  # nearly so
    o[k == 9] = 0.0
    tmin[k == 10] = -3.0
    tmin[k == 11] = 0.0
    tmax[k == 12] = np.inf
    tmax[k == 13] = -1.0
    tmax[k == 14] = np.nan
    d[k == 15] *= 1e20
    o[k == 16] *= 1e4
    tmax[k == 16] = 1e6
    d[k == 16] = -o[k == 16] / 7e4
    d[k == 17] = 0.0
    d[k == 18] *= 1e-6
    tmax[k == 18] *= 1e6
    # through the corner of a pile's bounds, past every triangle
    o[k == 19] = (0.95, 0.95, -3.0)
    d[k == 19] = (0.0005, 0.0007, 1.0)
    return np.concatenate([o, tmin[:, None], d, tmax[:, None]], 1).astype(np.float32)


@pytest.mark.parametrize("builder", [abi.BVH_SAH, abi.BVH_LBVH])
@pytest.mark.parametrize("n,kind", [(1, "soup"), (2, "soup"), (3, "soup"), (4, "flat"), (5, "soup"), (6, "flat"),
                                    (9, "soup"), (33, "flat"), (1500, "soup"), (4000, "flat"), (5000, "pile")])
def test_flags_equal_the_binary_walk(n, kind, builder):
    import risltc_amd
    import torch
    rng = np.random.default_rng(n)
    mesh = soup(n, kind, rng)
    ctx = risltc_amd.Context(0)
    ctx.set_bvh_builder(builder)
    ctx.set_scene(mesh, [[0.5] * 6])
    rays = rays_for(rng, 24 * 101 + 5)
    hits = torch.full((len(rays),), 7, dtype=torch.int32, device="cuda")
    ctx.trace_shadow_rays(torch.from_numpy(rays).cuda(), hits)
    torch.cuda.synchronize()
    L, bvh = orc.lib(), orc.OrcBvh()
    tri = np.ascontiguousarray(mesh.dequantized(), np.float32)
    (L.orc_bvh_build_sah if builder == abi.BVH_SAH else L.orc_bvh_build)(C.byref(bvh), orc.ptr(tri, orc.f32p), n)
    o, d = np.ascontiguousarray(rays[:, 0:3]), np.ascontiguousarray(rays[:, 4:7])
    want = np.array([L.orc_bvh_any_hit(C.byref(bvh), orc.ptr(o[i], orc.f32p), orc.ptr(d[i], orc.f32p),
                                       float(rays[i, 3]), float(rays[i, 7]), None) for i in range(len(rays))])
    L.orc_bvh_free(C.byref(bvh))
    got = hits.cpu().numpy()
    assert np.array_equal(got, want), np.flatnonzero(got != want)[:10] % 24
