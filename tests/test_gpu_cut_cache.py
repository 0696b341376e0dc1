"""The cache that a call of several tokens leaves behind when it is cut to the sinks and the window: its rows come from the old cache,
from the call's own tokens or from both, and so do the sinks.  Values bit for bit the tokens' own; keys those of a cache that was
fed in other pieces, up to the last bit of their rounding to bf16 (the angles of a tile follow from its first by recurrence)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _feed(kind, n_local, n_init, x, calls, H, Hkv, D):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    forward, rope, same = ATTN_FORWRAD[kind](n_local, n_init, fattn=False), RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t
    past, pos = None, 0
    for n in calls:
        q, k, v = (t[:, pos:pos + n] for t in x)
        _, past = forward(None, q, k, rope, True, past, same, same, lambda _: v, same, D, H, Hkv)
        pos += n
    return past


@pytest.mark.parametrize("kind", ["stream-llm", "infinite-lm"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n_local,n_init,calls", [
    (96, 16, [300]),                      # everything from one call
    (96, 16, [7, 200]),                   # sinks from both, the window from the call
    (96, 16, [150, 20, 33]),              # the window from both
    (96, 16, [112, 1, 40]),               # a full cache, a step, a short call
    (130, 0, [100, 100, 17, 200]),        # no sinks
    (64, 4, [500, 64, 65, 63])])          # calls about as long as the window
def test_rows_of_a_cut_cache(kind, D, n_local, n_init, calls):
    B, H, Hkv, T = 2, 4, 2, sum(calls)
    g = torch.Generator(device="cuda").manual_seed(T + D)
    x = [torch.randn((B, T, h * D), generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv)]
    past = _feed(kind, n_local, n_init, x, calls, H, Hkv, D)
    v = x[2].view(B, T, Hkv, D).permute(0, 2, 1, 3)
    assert torch.equal(past[1], torch.cat([v[:, :, :n_init], v[:, :, T - n_local:]], dim=2))
    ones = _feed(kind, n_local, n_init, x, [1] * T, H, Hkv, D)
    a, b = past[0].float(), ones[0].float()
    assert a.shape == b.shape and bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6).all())
