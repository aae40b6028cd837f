"""The two forms of the fast build's polygon integral (a wave whose polygons
are all unclipped with edges below 90 degrees, and the general form) give the
same bits: the compacted kernel and the per-lane debug kernel put different
candidates into a wave, so a polygon takes either form in the two."""
import numpy as np
import pytest

from risltc_amd import synth

pytestmark = pytest.mark.gpu


def lights(n, kind, count, rng):
    out = []
    for i in range(count):
        near = kind == "near" or (kind == "mixed" and i % 3 == 0)
        pts = synth.random_convex_polygon(rng, n)
        # near: metres wide and low over the ground, so that edges pass 90
        # degrees and the horizon cuts them; far: small and high above it
        size = rng.uniform(3.0, 9.0) if near else rng.uniform(0.05, 0.5)
        centre = rng.uniform([-8, -8, 0.2], [8, 8, 2.0]) if near else rng.uniform([-8, -8, 6.0], [8, 8, 12.0])
        out.append(synth.Light(pts, rng.uniform(0, 2 * np.pi, 3), centre, (size, size), rng.uniform(1, 10, 3)))
    return out


@pytest.mark.parametrize("n", [3, 4, 5, 7, 8])
@pytest.mark.parametrize("kind", ["near", "far", "mixed"])
def test_forms_agree(n, kind, ltc_table):
    import risltc_amd
    import torch
    base = synth.small_scene(seed=0, width=100, height=75, light_count=8)
    scene = synth.Scene("paths", base.mesh, base.materials, lights(n, kind, 40, np.random.default_rng(n)), base.camera,
                        100, 75, 2, 24, 0)
    ctx = risltc_amd.Context(0)
    ctx.load_scene(scene, *ltc_table)
    consts, s = ctx.frame_constants(noise_seed=n, animate=True), scene.settings()
    P = scene.width * scene.height
    vis = torch.empty(P, dtype=torch.int32, device="cuda")
    ctx.render_visibility(consts, vis)
    a, b = (torch.empty(P * 4, dtype=torch.float32, device="cuda") for _ in range(2))
    rec = torch.empty(P * 2 * 40, dtype=torch.float32, device="cuda")
    ctx.shade(consts, s, vis, a)
    ctx.shade_debug(consts, s, vis, b, rec)
    torch.cuda.synchronize()
    assert np.array_equal(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32))
    assert float(a.view(P, 4)[:, :3].std()) > 0.0
