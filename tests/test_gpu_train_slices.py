"""The training step's gradient at batches of seven slices of 2048 rows and
more, which its last kernel sums eight at a time with a remainder: each layer's
weights and each layer's biases against an FP64 backward pass rounded to bf16
at the same points (relative 2-norm below 1e-2 each, the bound that the step's
own test has for a layer as a whole). 65536 is the default batch."""
import numpy as np
import pytest

from test_gpu_learned import (PHI, bf16, forward, hash32, layer_bounds, layers, learned, learned_k1024,  # noqa: F401
                              learned_wide)

pytestmark = pytest.mark.gpu


def check(g, B):
    import torch
    ctx, spp, P = g["ctx"], 2, g["P"]
    out = torch.empty(P * 4, dtype=torch.float32, device="cuda")
    ctx.shade(g["consts"], g["scene"].settings(sample_count_light=spp, ris_candidate_count=8), g["vis"], out)
    cl = ctx.proposal_records()[0].cpu().numpy().view(np.uint32)
    before, _ = ctx.proposal_get_params()
    seed = 7 + B // 256
    ctx.proposal_train(g["consts"], g["vis"], batch=B, steps=1, lr=1e-4, seed=seed)
    _, grad = ctx.proposal_get_params()
    step_seed = (seed * PHI) & 0xFFFFFFFF
    items = hash32((step_seed * PHI + np.arange(B, dtype=np.uint64)) & 0xFFFFFFFF) % (P * spp)
    pix = (items // spp).astype(np.int64)
    vis = g["vis"].cpu().numpy().view(np.uint32)
    ok = ((vis[pix] >> 31) == 0) & (cl[items] != 0xFFFFFFFF)
    X = g["feats"][pix].astype(np.float64)
    H1, H2, H3, Z = forward(before, X)
    p = np.exp(Z - Z.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    p[np.arange(B), np.where(ok, cl[items], 0).astype(np.int64)] -= 1.0
    (W1, _), (W2, _), (W3, _), (W4, _) = layers(before)
    G4 = bf16((ok / ok.sum())[:, None] * p).astype(np.float64)
    G3 = bf16((G4 @ bf16(W4).astype(np.float64)) * (H3 > 0)).astype(np.float64)
    G2 = bf16((G3 @ bf16(W3).astype(np.float64)) * (H2 > 0)).astype(np.float64)
    G1 = bf16((G2 @ bf16(W2).astype(np.float64)) * (H1 > 0)).astype(np.float64)
    for l, ((G, A), (a, b)) in enumerate(zip(((G1, X), (G2, H1), (G3, H2), (G4, H3)),
                                             layer_bounds(W1.shape[0], W4.shape[0]))):
        w, bias = (G.T @ A).ravel(), G.sum(0)
        assert b - a == w.size + bias.size
        for name, got, ref in (("weights", grad[a:a + w.size], w), ("biases", grad[a + w.size:b], bias)):
            rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
            assert rel < 1e-2, (name, l + 1, B, rel)


@pytest.mark.parametrize("B", [14336, 16384, 16640, 65536])
def test_default_network(learned, B):  # noqa: F811
    check(learned, B)


@pytest.mark.parametrize("B", [16384, 18688])
def test_wide_network(learned_wide, B):  # noqa: F811
    check(learned_wide, B)


@pytest.mark.parametrize("B", [16640])
def test_many_outputs(learned_k1024, B):  # noqa: F811
    check(learned_k1024, B)
