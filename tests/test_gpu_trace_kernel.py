"""The persistent shadow-ray kernel (runs of rays, refills, walks shared by the
lanes of a draining wave, subtrees of a full stack) against the oracle's binary
walk, ray by ray: the debug records of frames over meshes on which its walks
are long, diverge or overflow, from a handful of rays to 40,000."""
import ctypes as C

import numpy as np
import pytest

import orc
from risltc_amd import abi, synth

pytestmark = pytest.mark.gpu


def mesh_of(kind, rng):
    if kind == "pile":  # every box on a path is met
        base = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.2], [0.0, 1.0, 0.2]])
        tri = 8.0 * (base[None] + rng.uniform(-1e-3, 1e-3, (1500, 3, 3))) - 4.0
    elif kind == "walls":  # boxes without extent
        tri = rng.uniform(-5, 5, (3000, 1, 3)) + rng.normal(0, 0.8, (3000, 3, 3))
        a = rng.integers(0, 3, 3000)
        tri[np.arange(3000), :, a] = tri[np.arange(3000), :1, a]
    elif kind == "cloud":  # stacks overflow
        tri = rng.uniform(-5, 5, (30000, 1, 3)) + rng.normal(0, 0.3, (30000, 3, 3))
    else:  # a few specks, origins far away: error bounds beyond whole nodes
        tri = rng.uniform(-1e-3, 1e-3, (7, 1, 3)) + rng.normal(0, 5e-4, (7, 3, 3))
    n = len(tri)
    return synth.Mesh(tri, np.tile(np.array([0.0, 0.0, 1.0]), (n, 3, 1)), np.zeros((n, 3, 2)), np.zeros(n, int),
                      np.zeros(n, int))


@pytest.mark.parametrize("builder", [abi.BVH_SAH, abi.BVH_LBVH])
@pytest.mark.parametrize("kind", ["pile", "walls", "cloud", "specks"])
def test_flags_equal_the_binary_walk(kind, builder, ltc_table):
    import risltc_amd
    import torch
    rng = np.random.default_rng(len(kind))
    base = synth.small_scene(seed=0, light_count=64)
    mesh = mesh_of(kind, rng)
    L, bvh = orc.lib(), orc.OrcBvh()
    dq = np.ascontiguousarray(mesh.dequantized(), np.float32)
    (L.orc_bvh_build_sah if builder == abi.BVH_SAH else L.orc_bvh_build)(C.byref(bvh), orc.ptr(dq, orc.f32p), len(dq))
    ctx = risltc_amd.Context(0)
    traced = 0
    try:
        ctx.set_bvh_builder(builder)
        ctx.load_scene(base, *ltc_table)
        ctx.set_scene(mesh, [[0.5] * 6])
        for width, height, spp, refill in ((3, 1, 1, 16), (61, 5, 1, 16), (200, 90, 1, 64), (200, 90, 2, 1)):
            P = width * height
            ctx.set_tuning(trace_refill=refill)
            k = risltc_amd.write_frame_constants(base.camera, width, height, mesh.dequantization_factor,
                                                 mesh.dequantization_summand, ctx.ltc_constants, noise_seed=P)
            vis = torch.from_numpy(rng.integers(0, len(dq), P).astype(np.int32)).cuda()
            out = torch.empty(P * 4, dtype=torch.float32, device="cuda")
            rec = torch.zeros(P * spp * abi.SAMPLE_RECORD_FLOATS, dtype=torch.float32, device="cuda")
            s = abi.default_settings(sample_count_light=spp, ris_candidate_count=4)
            ctx.shade_debug(k, s, vis, out, rec)
            torch.cuda.synchronize()
            r = rec.cpu().numpy().reshape(-1, abi.SAMPLE_RECORD_FLOATS)
            for t in range(2):
                state = r[:, abi.REC_STATE + t].view(np.uint32)
                at = np.flatnonzero((state == 2) | (state == 3))
                o = np.ascontiguousarray(r[at, abi.REC_POS:abi.REC_POS + 3])
                d = np.ascontiguousarray(r[at, abi.REC_DIR + 3 * t:abi.REC_DIR + 3 * t + 3])
                want = [L.orc_bvh_any_hit(C.byref(bvh), orc.ptr(o[i], orc.f32p), orc.ptr(d[i], orc.f32p), 1.0e-3,
                                          float(r[at[i], abi.REC_TMAX + t]), None) for i in range(len(at))]
                bad = np.flatnonzero((state[at] == 2) != (np.array(want, np.int64) == 1))
                assert bad.size == 0, (width, height, spp, refill, t, bad[:10])
                traced += len(at)
    finally:
        ctx.close()
        L.orc_bvh_free(C.byref(bvh))
    assert traced > 3000
