"""The resolve's counts for the visibility cache where a work-group's pixels
share few (cell, slot) pairs, and where they have more of them than its table
holds (cells far smaller than a pixel's footprint, 16 samples per pixel): the
counts equal those of the debug records exactly."""
import numpy as np
import pytest

from risltc_amd import abi
from test_gpu_learned import learned  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2_cells,cell,spp", [(0, 100.0, 3), (4, 50.0, 1), (16, 0.002, 1), (16, 0.002, 16),
                                                  (18, 0.0005, 5)])
def test_counts_equal_the_records(learned, log2_cells, cell, spp):  # noqa: F811
    import torch
    g = learned
    sc, ctx, P = g["scene"], g["ctx"], g["P"]
    if log2_cells:
        ctx.proposal_cache(log2_cells, cell, 2.0, True)
    else:
        ctx.proposal_cache(1, cell, 2.0, False)
    try:
        s = sc.settings(sample_count_light=spp, ris_candidate_count=8, proposal=abi.PROPOSAL_UNIFORM)
        out = torch.empty(P * 4, dtype=torch.float32, device="cuda")
        rec = torch.zeros(P * spp * abi.SAMPLE_RECORD_FLOATS, dtype=torch.float32, device="cuda")
        ctx.shade_debug(ctx.frame_constants(noise_seed=9, animate=True), s, g["vis"], out, rec)
        torch.cuda.synchronize()
        got = ctx.proposal_cache_read()
    finally:
        ctx.proposal_cache(0)
    r = rec.cpu().numpy().reshape(-1, abi.SAMPLE_RECORD_FLOATS)
    li = r[:, abi.REC_LIGHT].view(np.int32)
    st = r[:, abi.REC_STATE:abi.REC_STATE + 2].view(np.uint32)
    hit, miss = (st == 2).sum(1), (st == 3).sum(1)
    ok = (li >= 0) & (hit + miss > 0)
    key = r[ok, abi.REC_CACHE_KEY].view(np.uint32).astype(np.int64)
    slot = (li[ok] if log2_cells else g["col"][li[ok]]).astype(np.int64)
    want = np.zeros(got.shape, dtype=np.int64)
    np.add.at(want, (key, slot, 0), miss[ok])
    np.add.at(want, (key, slot, 1), hit[ok])
    assert ok.sum() > 0.2 * P
    if spp == 16:  # more pairs per 256 pixels than the table's 1024
        assert np.unique(key * got.shape[1] + slot).size > 1024 * P / 256
    assert np.array_equal(got.astype(np.int64), want)
