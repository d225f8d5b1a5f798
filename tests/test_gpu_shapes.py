"""Kernels at the sizes where their tilings can go wrong (partial tiles, remainders, the smallest and
largest of a dispatch's range), against the oracle under the reference's per-kernel tolerance."""
import numpy as np
import pytest

from ops_lib import Prog, fast_values, within
from test_gpu_ops import both

pytestmark = pytest.mark.gpu


def attention_case(ctx, oracle, B, L, S, H, heads):
    """Attention and its three gradients, random masked keys: results, oracle's, mask and bound."""
    q, G = (fast_values(s, B * L * H, 0.5).reshape(B * L, H) for s in (12, 15))
    k, v = (fast_values(s, B * S * H, 0.5).reshape(B * S, H) for s in (13, 14))
    mask = (np.random.default_rng(S).random((B, S)) < 0.7).astype(np.float32)
    mask[:, S // 2] = 1.0
    p = Prog()
    qi, ki, vi = p.input("q", (B * L, H)), p.input("k", (B * S, H)), p.input("v", (B * S, H))
    mi, Gi = p.input("mask", (B, S)), p.input("G", (B * L, H))
    attr = f"[heads = {heads}]"
    outs = [p.op("Attention", [qi, ki, vi, mi], (B * L, H), attr)]
    for op, rows in (("AttentionGradQ", B * L), ("AttentionGradK", B * S), ("AttentionGradV", B * S)):
        outs.append(p.op(op, [qi, ki, vi, mi, Gi], (rows, H), attr))
    got, want = both(ctx, oracle, p.out(*outs), {"q": q, "k": k, "v": v, "mask": mask, "G": G}, (0, 1, 2, 3))
    # r: sum over keys of |p| |v|-like terms, bounded by the largest row magnitudes.
    scale = np.abs(v).max() + np.abs(G).max() * (np.abs(q).max() + np.abs(k).max()) * np.sqrt(H // heads) * 2
    return got, want, mask, scale


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("B,L,S,H,heads", [
    (1, 1, 1, 16, 1), (2, 15, 15, 32, 2), (2, 17, 17, 64, 1), (3, 100, 100, 192, 3), (1, 150, 150, 64, 1),
    (2, 33, 33, 128, 1),     # head width 128: two-wave blocks, tiles of 32 rows
    (3, 300, 300, 32, 2),    # several streamed tiles, the last of 44 rows
    (43, 100, 100, 224, 14),  # over 4096 row tiles: four-wave blocks streaming 32-row tiles
    (2, 20, 48, 64, 2),      # fewer queries than keys, whole key tiles
])
def test_attention_over_partial_tiles(ctx, oracle, B, L, S, H, heads, mixed):
    """Row counts that are no multiple of 16, in f32 also under mixed precision: rows past the end
    take no part and are not written, masked keys' gradients are +0."""
    ctx.set_precision(mixed)
    try:
        got, want, mask, scale = attention_case(ctx, oracle, B, L, S, H, heads)
    finally:
        ctx.set_precision(False)
    for idx, (g, w) in enumerate(zip(got, want)):
        ok, worst = within(g, w, np.abs(w) + scale)
        assert ok, (idx, worst)
    for g in (got[2], got[3]):
        assert np.all(g.reshape(B * S, H)[mask.reshape(-1) == 0] == 0)
