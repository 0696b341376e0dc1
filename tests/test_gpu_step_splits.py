"""A step's workgroups of eight waves at the edges of what they take: caches of a block of 16 keys, a block of every wave, and one key more
or fewer, so that the step's own key is a block of its own to any wave; heads and batch rows for a split each, several, and more workgroups
than the chip has places for.

Against a dense softmax in 64 bits over the cache that the type returns, as in the test of the joins and with its bound: partial rows are fp16
(a relative 2^-11) and the result bf16 (2^-9), within 1e-2 of a row's largest value."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,D,B", [(8, 2, 128, 1), (6, 3, 128, 1), (2, 2, 128, 2), (10, 2, 64, 1), (2, 1, 64, 1), (3, 3, 64, 1), (40, 40, 128, 7), (36, 36, 64, 15)])
@pytest.mark.parametrize("past", [14, 15, 16, 126, 127, 128, 142, 255, 400])
def test_steps_at_the_edges_of_their_splits(H, Hkv, D, B, past):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    g = torch.Generator(device="cuda").manual_seed(past + H)
    rand = lambda n, h: torch.randn((B, n, h * D), generator=g, device="cuda").bfloat16()
    forward, rope, same = ATTN_FORWRAD["origin"](False), RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t
    call = lambda q, k, v, cache: forward(None, q, k, rope, True, cache, same, same, lambda _: v, same, D, H, Hkv)
    _, cache = call(rand(past, H), rand(past, Hkv), rand(past, Hkv), None)
    for _ in range(2):
        q = rand(1, H)
        out, cache = call(q, rand(1, Hkv), rand(1, Hkv), cache)
        k, v = (t.double().repeat_interleave(H // Hkv, dim=1) for t in cache[:2])
        n = k.shape[2]
        angle = (n - 1) * rope.inv_freq.double().cuda()
        cos, sin = (torch.cat([f(angle), f(angle)]) for f in (torch.cos, torch.sin))
        x = q.view(B, 1, H, D).permute(0, 2, 1, 3).double()
        rot = (x * cos + torch.cat([-x[..., D // 2:], x[..., :D // 2]], -1) * sin).bfloat16().double()
        p = torch.softmax((rot * k).sum(-1) / math.sqrt(D), -1)
        want = (p[..., None] * v).sum(2)
        assert float(((out.view(B, H, D).double() - want).abs().amax(-1) / want.abs().amax(-1)).max()) <= 1e-2
