"""Workgroups that stage the rows of several kv heads (fewer than three query heads each, more workgroups than the chip holds at once):
the rows of the same call one kv head at a time, whose workgroups take one, at ragged lengths and where the last group is not full."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 5, 5, 64, 3317), (1, 6, 3, 64, 5475), (2, 3, 3, 128, 2741), (1, 10, 5, 128, 3313), (1, 9, 9, 64, 1841)]


def same_rotation(got, want):
    """x cos - y sin in fp32 with either product joined to the sum (2^-23 of |x| + |y| < 16), then one rounding to bf16 (2^-7 between
    neighbours)."""
    got, want = got.float(), want.float()
    return bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -19).all())


@pytest.mark.parametrize("B,H,Hkv,D,n", SIZES)
def test_ingest_of_several_heads(B, H, Hkv, D, n):
    from infllm_amd import ops
    G, cap, pos0, tiles = H // Hkv, n + 70, 123456, (n + 15) // 16
    assert tiles * B * Hkv > 1024 >= tiles
    g = torch.Generator(device="cuda").manual_seed(n)
    bf = lambda h: torch.randn((B, n, h, D), generator=g, device="cuda").bfloat16().transpose(1, 2)
    q, k, v = bf(H), bf(Hkv), bf(Hkv)
    inv_freq = 1.0 / 1e4 ** (torch.arange(0, D, 2, device="cuda").float() / D)

    def ingest(b, hs, gs):
        z = lambda h, rows: torch.zeros((b.stop - b.start, h, rows, D), dtype=torch.bfloat16, device="cuda")
        h, hkv = hs.stop - hs.start, gs.stop - gs.start
        outs = [z(hkv, cap), z(hkv, cap), z(hkv, cap), torch.ones((b.stop - b.start, h, cap), device="cuda"), z(h, n), z(h, n),
                torch.full((b.stop - b.start, tiles, h * D), 9.0, device="cuda")]
        ops.ingest(q[b, hs], k[b, gs], v[b, gs], pos0, 4095, inv_freq, 1.0, *outs)
        return outs[:6] + [outs[6].view(-1, tiles, h, D).transpose(1, 2)]
    together = ingest(slice(0, B), slice(0, H), slice(0, Hkv))
    for b in range(B):
        for i in range(Hkv):
            hs, gs = slice(i * G, i * G + G), slice(i, i + 1)
            for j, (got, want) in enumerate(zip(together, ingest(slice(b, b + 1), hs, gs))):
                got = got[b:b + 1, gs if j < 3 else hs]          # rings of raw keys, rotated keys, values, scores; queries; sums of 16 of them
                if j == 6:
                    assert float((got - want).abs().max()) <= 16 * 2.0 ** -19, (b, i)
                else:
                    assert same_rotation(got, want) if j in (1, 4, 5) else torch.equal(got, want), (b, i, j)


@pytest.mark.parametrize("kind", ["origin", "stream-llm", "infinite-lm"])
@pytest.mark.parametrize("B,H,Hkv,D,n", SIZES)
def test_window_rows_of_several_heads(B, H, Hkv, D, n, kind):
    """The caches of two calls: rotated keys, values, the sinks kept beside them.  (The outputs' key splits depend on the heads.)"""
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    g, G = torch.Generator(device="cuda").manual_seed(n), H // Hkv
    q, k, v = (torch.randn((B, 2 * n, h, D), generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv))
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](n - 100, 40, fattn=False)
    rope, same = RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t

    def calls(b, hs, gs):
        past, out = None, []
        for sl in (slice(0, n), slice(n, 2 * n)):
            rows = [t[b, sl, heads].flatten(2) for t, heads in ((q, hs), (k, gs), (v, gs))]
            o, past = forward(None, rows[0], rows[1], rope, True, past, same, same, lambda _: rows[2], same, D, hs.stop - hs.start, gs.stop - gs.start)
            out.append(o.view(o.shape[0], n, -1, D).transpose(1, 2))
        return out, [t for t in past if torch.is_tensor(t)]
    outs, cache = calls(slice(0, B), slice(0, H), slice(0, Hkv))
    for b in range(B):
        for i in range(Hkv):
            hs, gs = slice(i * G, i * G + G), slice(i, i + 1)
            want_outs, want_cache = calls(slice(b, b + 1), hs, gs)
            assert len(cache) == len(want_cache) >= 2
            for j, (got, want) in enumerate(zip(cache, want_cache)):
                got = got[b:b + 1, gs]
                assert torch.equal(got, want) if j else same_rotation(got, want), (b, i, j)
            # Both results are rounded to bf16, 2^-8 of an element each at most and a third of that in the mean square: what is left of
            # 2^-7 is for probabilities and partial rows that were rounded under another maximum (a row with few keys: 2^-9 of a weight)
            for got, want in zip(outs, want_outs):
                assert float((got[b:b + 1, hs].float() - want.float()).norm()) <= 2.0 ** -7 * float(want.float().norm()), (b, i)
