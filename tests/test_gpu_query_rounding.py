"""Queries are rounded once, as rotated rows: the softmax scale is applied to their products, in 32 bits.  Angles are 0 here, so that queries
of 1.0 stay exact, as do all products; a key far below the others makes a rounding of scaled queries (0.3 % of 1 / sqrt(128) x log2(e))
one of 0.3 % of its logit, 14 % of its probability.

The row of a query is that key's probability times its value, a power of two near the probability's inverse.  It is rounded to bf16 as a
probability and as an output (half of 2^-7, the step of 8 significant bits, each) and to fp16 in a partial row (2^-11): 8.3e-3 of it."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["origin", "infinite-lm", "stream-llm"])
@pytest.mark.parametrize("H,Hkv,D", [(8, 2, 128), (3, 3, 128), (8, 2, 64), (3, 3, 64), (4, 2, 80)])
@pytest.mark.parametrize("n", [2, 70, 1500])
def test_products_are_scaled_not_queries(kind, H, Hkv, D, n):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    n_local, n_init, low, same = 40, 4, 4.0 * math.sqrt(D), lambda t: t
    total = n + 1                                                               # a prompt, and a step behind it
    k, v = torch.zeros(1, total, Hkv, D), torch.zeros(1, total, Hkv, D)
    far = torch.arange(total) % 30 == 1                                         # (one of the sinks, and one in every window of 40)
    k[:, far], v[:, far] = -4.0, 2.0 ** round(low / math.log(2))
    dist = torch.arange(total)[:, None] - torch.arange(total)[None, :]
    seen = dist >= 0
    if kind != "origin":
        seen &= (dist < n_local) | (torch.arange(total)[None, :] < n_init)
    p = torch.where(far, -low, 0.0).double().expand(total, total).masked_fill(~seen, -torch.inf).softmax(-1)
    want = (p @ v[0].flatten(1).double()).view(total, Hkv, D).repeat_interleave(H // Hkv, 1).flatten(1)
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](n_local, n_init, fattn=False)
    rope, past = RotaryEmbeddingESM(D, distance_scale=0.0, device="cuda"), None
    kd, vd = (t.bfloat16().flatten(2).cuda() for t in (k, v))
    for a, b in ((0, n), (n, total)):
        rows = torch.ones(1, b - a, H * D, dtype=torch.bfloat16, device="cuda")
        got, past = forward(None, rows, kd[:, a:b], rope, True, past, same, same, lambda _: vd[:, a:b], same, D, H, Hkv)
        off = (got[0].cpu().double() - want[a:b]).abs() / want[a:b].clamp_min(1e-30)
        assert float(off.max()) <= 8.4e-3, (a, b, float(off.max()))
