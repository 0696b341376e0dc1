"""A step of the sliding-window and causal types as one launch against the launch in front and the attention (no tickets given): the
first token, old rows in place and copied, caches that are cut, sinks that are still being collected, groups of one to eight heads,
several batch rows.  Caches bit for bit; outputs within the rounding of fp16 partial rows at other split boundaries and of the result
to bf16 (2^-7 of a row's largest value)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,past", [("origin", 0), ("origin", 1), ("origin", 700), ("stream-llm", 0), ("stream-llm", 90), ("stream-llm", 700),
                                       ("infinite-lm", 3), ("infinite-lm", 111), ("infinite-lm", 112), ("infinite-lm", 700)])
@pytest.mark.parametrize("H,Hkv,D,B", [(4, 4, 128, 1), (6, 2, 64, 2), (16, 2, 128, 1), (8, 4, 64, 3)])
def test_one_launch_is_the_two(kind, past, H, Hkv, D, B, monkeypatch):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM, _sink_window
    g = torch.Generator(device="cuda").manual_seed(past + H)
    x = [torch.randn((B, past + 4, h * D), generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv)]
    same = lambda t: t

    def stream():
        forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](96, 16, fattn=False)
        rope, cache, outs = RotaryEmbeddingESM(D, base=1e4, device="cuda"), None, []
        for lo, hi in ([(0, past)] if past else []) + [(past + i, past + i + 1) for i in range(4)]:
            q, k, v = (t[:, lo:hi] for t in x)
            out, cache = forward(None, q, k, rope, True, cache, same, same, lambda _: v, same, D, H, Hkv)
            outs.append(out)
        return outs, cache
    got, cache = stream()
    monkeypatch.setattr(_sink_window, "_ticket", lambda *_: 0)
    want, other = stream()
    assert torch.equal(cache[0], other[0]) and torch.equal(cache[1], other[1])
    if kind == "infinite-lm":
        assert torch.equal(cache[3], other[3])
    for a, b in zip(got, want):
        a, b = (t.view(B, -1, H, D).float() for t in (a, b))
        assert bool(((a - b).abs().amax(-1) <= 2.0 ** -7 * b.abs().amax(-1)).all())


@pytest.mark.parametrize("kind", ["stream-llm", "infinite-lm"])
@pytest.mark.parametrize("n_local", [64, 65, 66, 256, 257, 258, 700])          # rows copied: one fewer, in pieces of 64 or 256
@pytest.mark.parametrize("H,Hkv,D,B", [(4, 4, 128, 1), (16, 1, 128, 2), (6, 3, 64, 2)])
def test_copies_of_a_full_cache(kind, n_local, H, Hkv, D, B, monkeypatch):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM, _sink_window
    n_init, T = 5, n_local + 9
    g = torch.Generator(device="cuda").manual_seed(T)
    x = [torch.randn((B, T, h * D), generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv)]
    same = lambda t: t

    def stream():
        forward, rope, cache = ATTN_FORWRAD[kind](n_local, n_init, fattn=False), RotaryEmbeddingESM(D, base=1e4, device="cuda"), None
        for lo, hi in [(0, T - 4)] + [(i, i + 1) for i in range(T - 4, T)]:
            q, k, v = (t[:, lo:hi] for t in x)
            out, cache = forward(None, q, k, rope, True, cache, same, same, lambda _: v, same, D, H, Hkv)
        return out, cache
    got, cache = stream()
    monkeypatch.setattr(_sink_window, "_ticket", lambda *_: 0)
    want, other = stream()
    assert torch.equal(cache[0], other[0]) and torch.equal(cache[1], other[1])
    v = x[2].view(B, T, Hkv, D).permute(0, 2, 1, 3)
    assert torch.equal(cache[1], torch.cat([v[:, :, :n_init], v[:, :, T - n_local:]], dim=2))
    a, b = (t.view(B, H, D).float() for t in (got, want))
    assert bool(((a - b).abs().amax(-1) <= 2.0 ** -7 * b.abs().amax(-1)).all())
