"""Tables of 256 constant logits with NaN at fixed places of a lane's groups of
four: one, a pair in each position, three, all four, in several groups of every
lane. A NaN is never kept and does not hide the other logits of its group, nor
those of the other groups."""
import math

import numpy as np
import pytest

from risltc_amd import abi, synth
from test_gpu_learned import layer_bounds, table_slots

pytestmark = pytest.mark.gpu

PLACES = [(2, 3), (0, 1), (0, 1, 2, 3), (1, 3), (0, 2), (3,), (1, 2, 3), (0, 3), (1, 2)]


@pytest.mark.parametrize("width", [64, 128])
@pytest.mark.parametrize("turn", range(4))
def test_nan_in_groups(ltc_table, width, turn):
    import risltc_amd
    import torch
    sc = synth.small_scene(seed=4, width=64, height=48, light_count=1200)
    ctx = risltc_amd.Context(0)
    try:
        ctx.load_scene(sc, *ltc_table)
        assert set(np.unique(ctx.cluster_lights(256, 5))) == set(range(256))  # none is empty
        ctx.proposal_init(3, width=width, outputs=256)
        params, _ = ctx.proposal_get_params()
        (a3, _), (a4, b4) = layer_bounds(width, 256)[2:]
        params[a3:] = 0.0
        # lane group g ranks outputs 16 t + 4 g + i; its best four are spread
        # over tiles, some of them beside a NaN
        bias = np.random.default_rng(turn).choice(np.float32([-1, -3, -3, -3]), 256)
        bias[16 * np.arange(16) + 5 * turn % 16] = 0.0
        for t in range(16):
            for g in range(4):
                if (t + g + turn) % 3 != 0:
                    bias[[16 * t + 4 * g + i for i in PLACES[(t + 2 * g + turn) % len(PLACES)]]] = np.nan
        params[b4 - 256:b4] = bias
        ctx.proposal_set_params(params)
        top = np.nanmax(bias)
        ids, weights = np.zeros(16, np.int64), np.zeros(16, np.int64)
        for g in range(4):
            own = [c for c in range(256) if c % 16 // 4 == g and not np.isnan(bias[c])]
            for s, c in enumerate(sorted(own, key=lambda c: (-bias[c], c))[:4]):
                ids[4 * g + s], weights[4 * g + s] = c, int(255 * math.exp(bias[c] - top) + 0.5)
        w, h = 67, 5
        consts = ctx.frame_constants()
        consts.viewport_size[0], consts.viewport_size[1] = w, h
        vis = torch.arange(w * h, dtype=torch.int32, device="cuda") % sc.mesh.triangle_count
        table = torch.full((w * h * abi.proposal_table_bytes(256),), 9, dtype=torch.uint8, device="cuda")
        ctx.proposal_update(consts, vis, table)
        torch.cuda.synchronize()
        gi, gw = table_slots(table.cpu().numpy().reshape(w * h, -1), 256)
        assert np.array_equal(gw, np.broadcast_to(weights, gw.shape))
        assert np.array_equal(gi, np.broadcast_to(ids, gi.shape))
    finally:
        ctx.close()
