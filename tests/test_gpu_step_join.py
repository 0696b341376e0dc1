"""A step of the sliding-window and causal types joins its key splits in the launch that makes them: one split to 64, heads that share
a key head alone, in pairs, threes, fours and more, heads of 64 and 128, several batch rows, steps one after the other (the
tickets are zero again behind each).

Against a dense softmax in 64 bits over the cache that the type returns.  Partial rows are fp16 (a relative 2^-11) and the result
bf16 (2^-9): within 1e-2 of a row's largest value."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,D", [(1, 1, 128), (4, 2, 128), (6, 2, 64), (8, 2, 128), (16, 2, 64), (12, 12, 64), (32, 8, 128)])
@pytest.mark.parametrize("past,B", [(1, 1), (40, 2), (700, 3), (9000, 1)])
def test_steps_of_the_causal_type(H, Hkv, D, past, B):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    g = torch.Generator(device="cuda").manual_seed(past + H)
    rand = lambda n, h: torch.randn((B, n, h * D), generator=g, device="cuda").bfloat16()
    forward, rope, same = ATTN_FORWRAD["origin"](False), RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t
    call = lambda q, k, v, cache: forward(None, q, k, rope, True, cache, same, same, lambda _: v, same, D, H, Hkv)
    _, cache = call(rand(past, H), rand(past, Hkv), rand(past, Hkv), None)
    for _ in range(3):
        q = rand(1, H)
        out, cache = call(q, rand(1, Hkv), rand(1, Hkv), cache)
        k, v = (t.double().repeat_interleave(H // Hkv, dim=1) for t in cache[:2])
        n = k.shape[2]
        # the query at position n - 1, rotated as the type rotates it (bf16), against the rotated keys of the cache
        angle = (n - 1) * rope.inv_freq.double().cuda()
        cos, sin = (torch.cat([f(angle), f(angle)]) for f in (torch.cos, torch.sin))
        x = q.view(B, 1, H, D).permute(0, 2, 1, 3).double()
        rot = (x * cos + torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1) * sin).bfloat16().double()
        p = torch.softmax((rot * k).sum(-1) / math.sqrt(D), -1)
        want = (p[..., None] * v).sum(2)
        got = out.view(B, H, D).double()
        assert float(((got - want).abs().amax(-1) / want.abs().amax(-1)).max()) <= 1e-2
