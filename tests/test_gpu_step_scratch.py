"""Steps of the sliding-window and causal types that take their scratch from the cache they continue (up to 4 MiB of it: 244 query rows
of 128) against steps from copies of that cache, which bring none and work in two launches: within the rounding of fp16 partial rows at
other split boundaries and of the result to bf16 (2^-7 of a row's largest value), also where two continuations share a cache."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,B,H,Hkv,D", [("stream-llm", 1, 4, 2, 128), ("stream-llm", 61, 4, 4, 128), ("origin", 62, 4, 2, 128), ("infinite-lm", 8, 32, 8, 128),
                                            ("origin", 3, 36, 36, 64), ("stream-llm", 2, 4, 2, 32)])
def test_steps_with_the_scratch_of_their_cache(kind, B, H, Hkv, D):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    g, past = torch.Generator(device="cuda").manual_seed(B), 150
    x = [torch.randn((B, past + 4, h * D), generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv)]
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](96, 16, fattn=False)
    rope, same = RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t

    def call(lo, hi, cache):
        q, k, v = (t[:, lo:hi] for t in x)
        return forward(None, q, k, rope, True, cache, same, same, lambda _: v, same, D, H, Hkv)
    _, cache = call(0, past, None)
    for i in range(past, past + 4):
        bare = tuple(t.clone() if torch.is_tensor(t) else t for t in cache)
        want, _ = call(i, i + 1, bare)
        first, going_on = call(i, i + 1, cache)
        second, _ = call(i, i + 1, cache)
        want = want.view(B, H, D).float()
        for out in (first, second):
            assert bool(((out.view(B, H, D).float() - want).abs().amax(-1) <= 2.0 ** -7 * want.abs().amax(-1)).all())
        cache = going_on
