"""Proposal tables at view sizes around a wave's 64 pixels, a work-group's 256
and a full launch, for each network shape, with an output layer of constant
logits: the logits are the biases exactly, so the tables follow from them.
Biases of few values tie; some are NaN (never kept); the clusters past the
count are empty. Biases of 0, -1 and -3 give weights 255, 94 and 13, well
inside their rounding, so the tables are compared exactly."""
import math

import numpy as np
import pytest

from risltc_amd import synth
from test_gpu_learned import group_values, layer_bounds, table_slots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,outputs,K", [(64, 256, 200), (128, 256, 256), (64, 1024, 600), (128, 1024, 700)])
def test_tables_of_constant_logits(ltc_table, width, outputs, K):
    import risltc_amd
    import torch
    from risltc_amd import abi
    sc = synth.small_scene(seed=4, width=64, height=48, light_count=1200)
    ctx = risltc_amd.Context(0)
    try:
        ctx.load_scene(sc, *ltc_table)
        col = ctx.cluster_lights(K, 5)
        ctx.proposal_init(3, width=width, outputs=outputs)
        params, _ = ctx.proposal_get_params()
        rng = np.random.default_rng(width + outputs)
        (a3, _), (a4, b4) = layer_bounds(width, outputs)[2:]
        params[a3:] = 0.0  # the last hidden layer and the output weights
        quad = outputs // 256
        bias = rng.choice(np.float32([0, -1, -3, -3, -3]), 256).repeat(quad)
        bias[rng.choice(256, 5, replace=False) * quad] = np.nan  # a quad with one is not kept
        params[b4 - outputs:b4] = bias
        ctx.proposal_set_params(params)
        v, lane_group, live = group_values(bias.astype(np.float64), np.bincount(col, minlength=outputs), outputs)
        live = live & ~np.isnan(v)
        top = v[live].max()
        ids, weights, slack = np.zeros(16, np.int64), np.zeros(16, np.int64), np.zeros(16, np.int64)
        for g in range(4):
            for s, c in enumerate(sorted(np.flatnonzero(live & (lane_group == g)), key=lambda c: (-v[c], c))[:4]):
                e = 255 * math.exp(v[c] - top) + 0.5
                weights[4 * g + s] = int(e)
                slack[4 * g + s] = abs(e - round(e)) < 1e-3  # half of a quad's clusters empty: 127.5
                ids[4 * g + s] = c if weights[4 * g + s] else 0
        for w, h in ((1, 1), (63, 1), (64, 1), (65, 3), (257, 1), (401, 331)):
            consts = ctx.frame_constants()
            consts.viewport_size[0], consts.viewport_size[1] = w, h
            vis = torch.from_numpy(rng.integers(0, sc.mesh.triangle_count, w * h).astype(np.int32)).cuda()
            vis[::7] = -1
            table = torch.full((w * h * abi.proposal_table_bytes(outputs),), 9, dtype=torch.uint8, device="cuda")
            # an address that is a multiple of four only
            logits = torch.zeros(w * h * outputs + 2, dtype=torch.float32, device="cuda")[1:-1]
            ctx.proposal_update(consts, vis, table, logits)
            torch.cuda.synchronize()
            got = logits.cpu().numpy().reshape(-1, outputs)
            assert np.array_equal(got, np.broadcast_to(bias, got.shape), equal_nan=True), (w, h)
            shaded = vis.cpu().numpy() >= 0
            gi, gw = table_slots(table.cpu().numpy().reshape(w * h, -1), outputs)
            assert np.all(gw[~shaded] == 0), (w, h)
            assert np.all(np.abs(gw[shaded] - weights) <= slack), (w, h)
            assert np.array_equal(gi[shaded], np.broadcast_to(ids, gi[shaded].shape)), (w, h)
    finally:
        ctx.close()
