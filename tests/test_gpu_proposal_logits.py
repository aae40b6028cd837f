"""Logits of the networks with 1024 outputs at views around a wave's 64 pixels,
where the last group of pixels is partly outside: the same bits as the first
rows of a view in which those groups are whole, and nothing written past the
view. (The values are checked in test_gpu_learned.)"""
import numpy as np
import pytest

from risltc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [64, 128])
def test_logits_of_partial_groups(ltc_table, width):
    import risltc_amd
    import torch
    sc = synth.small_scene(seed=4, width=64, height=48, light_count=1200)
    ctx = risltc_amd.Context(0)
    try:
        ctx.load_scene(sc, *ltc_table)
        ctx.cluster_lights(1024, 2)
        ctx.proposal_init(width, width=width, outputs=1024)
        rng = np.random.default_rng(width)

        def logits(w, h, vis):
            consts = ctx.frame_constants()
            consts.viewport_size[0], consts.viewport_size[1] = w, h
            room = torch.full((w * h * 1024 + 1 + 4096,), 12345.0, dtype=torch.float32, device="cuda")
            ctx.proposal_update(consts, vis[:w * h].contiguous(), None, room[1:])  # an address that is a multiple of four
            torch.cuda.synchronize()
            got = room.cpu().numpy()
            assert got[0] == 12345.0 and np.all(got[1 + w * h * 1024:] == 12345.0), (w, h)
            return got[1:1 + w * h * 1024].view(np.uint32).reshape(w * h, 1024)

        for w, h in ((1, 1), (7, 1), (8, 1), (63, 1), (64, 1), (65, 1), (43, 3), (64, 5), (251, 7)):
            vis = torch.from_numpy(rng.integers(0, sc.mesh.triangle_count, w * (h + 64)).astype(np.int32)).cuda()
            whole, part = logits(w, h + 64, vis), logits(w, h, vis)
            assert np.array_equal(part, whole[:w * h]), (w, h)
            if w * h > 64:
                assert np.unique(part[:, 0]).size > 8  # pixels differ
    finally:
        ctx.close()
