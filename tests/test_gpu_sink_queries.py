"""Queries that the attention rotates to the sinks' angle itself: more sinks than a key split has tiles (splits that begin among the
sinks, that cross into them, that see none), calls that are no whole tile of queries, rows of the projection apart or next to each
other - the same bits either way, and oracle.siblings' results (2e-2 / 2e-3, the bounds of the other tests of these types)."""
import pytest
import torch

from oracle.rope import RopeOracle
from oracle.siblings import SinkWindowOracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["stream-llm", "infinite-lm"])
@pytest.mark.parametrize("D,H,Hkv,B", [(128, 4, 2, 1), (64, 6, 3, 2), (128, 5, 1, 2), (64, 4, 4, 1), (128, 8, 2, 2), (128, 9, 1, 1)])
@pytest.mark.parametrize("calls,n_local,n_init", [([400, 333, 33, 1, 2], 64, 200), ([65, 31, 290], 96, 65), ([700], 500, 64)])
def test_prompts_with_sinks(kind, D, H, Hkv, B, calls, n_local, n_init):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    T, g = sum(calls), torch.Generator().manual_seed(sum(calls) + D)
    wide = torch.randn(B, T, (H + 2 * Hkv) * D, generator=g).bfloat16()                 # one projection's output: q, k and v next to each other
    forward, rope, same = ATTN_FORWRAD[kind](n_local, n_init, fattn=False), RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t

    def run(q, k, v):
        past, outs, pos = None, [], 0
        for n in calls:
            rows = [t[:, pos:pos + n] for t in (q, k, v)]
            o, past = forward(None, rows[0], rows[1], rope, True, past, same, same, lambda _: rows[2], same, D, H, Hkv)
            outs.append(o)
            pos += n
        return torch.cat(outs, dim=1)
    apart = wide.cuda().split([H * D, Hkv * D, Hkv * D], dim=-1)
    got = run(*apart)
    assert torch.equal(got, run(*(t.contiguous() for t in apart)))
    heads = lambda t, h: t.reshape(B, T, h, D).permute(0, 2, 1, 3).float()
    x = [heads(t, h) for t, h in zip(wide.split([H * D, Hkv * D, Hkv * D], dim=-1), (H, Hkv, Hkv))]
    oracle, want, pos = SinkWindowOracle(RopeOracle(D, base=1e4), n_local, n_init, kind), [], 0
    for n in calls:
        want.append(oracle.append(*(t[:, :, pos:pos + n] for t in x)))
        pos += n
    err = (heads(got.cpu(), H) - torch.cat(want, dim=2)).abs()
    assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, (float(err.max()), float(err.mean()))


@pytest.mark.parametrize("kind", ["origin", "stream-llm", "infinite-lm"])
@pytest.mark.parametrize("B,H,Hkv,n", [(1, 32, 8, 4099), (2, 33, 3, 2000), (1, 8, 2, 37), (1, 8, 1, 513), (3, 4, 1, 64)])
def test_queries_rotated_where_they_are_attended(kind, B, H, Hkv, n):
    """Four query heads of 128 a kv head, or eight and more, whose attention rotates them, against the same heads in calls of one, whose
    queries are staged: a last tile that is not full, a second call behind a cache, rows apart from each other."""
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    D, G, g = 128, H // Hkv, torch.Generator(device="cuda").manual_seed(n)
    q, k, v = torch.randn((B, 2 * n, (H + 2 * Hkv) * D), generator=g, device="cuda").bfloat16().split([H * D, Hkv * D, Hkv * D], dim=-1)
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](n // 2, 70, fattn=False)
    rope, same = RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t

    def run(q, k, v, heads, kv_heads):
        past, outs = None, []
        for sl in (slice(0, n), slice(n, 2 * n)):
            rows = [t[:, sl] for t in (q, k, v)]
            o, past = forward(None, rows[0], rows[1], rope, True, past, same, same, lambda _: rows[2], same, D, heads, kv_heads)
            outs.append(o)
        return torch.cat(outs, dim=1)
    got = run(q, k, v, H, Hkv).view(B, 2 * n, H, D)
    for i in range(H):
        part = [t.reshape(B, 2 * n, -1, D)[:, :, j] for t, j in ((q, i), (k, i // G), (v, i // G))]
        want = torch.cat([run(*(t[b:b + 1] for t in part), 1, 1) for b in range(B)]).float()
        # results rounded to bf16, 2^-8 of an element each at most and a third of that in the mean square; the rest of 2^-7 for
        # probabilities, partial rows and single rotated elements that are rounded another way
        assert float((got[:, :, i].float() - want).norm()) <= 2.0 ** -7 * float(want.norm()), i


@pytest.mark.parametrize("kind", ["origin", "stream-llm", "infinite-lm"])
@pytest.mark.parametrize("off", [1, 2, 4, 8])
def test_queries_at_any_address(kind, off, monkeypatch):
    """Query rows that begin `off` elements behind a multiple of 16 bytes (a caller of the C function may have such): those of the calls
    whose attention would take them straight into LDS are staged, and the results differ as the two ways do."""
    from infllm_amd import _lib
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM, _sink_window
    B, H, Hkv, D, g = 1, 8, 2, 128, torch.Generator(device="cuda").manual_seed(off)
    calls, fields, lib = [333, 70], [n for n, _ in _lib.WindowArgs._fields_], _lib.load()
    x = [torch.randn((B, sum(calls), h * D), generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv)]
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](100, 30, fattn=False)
    rope, same, rooms = RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t, []

    class Moved:
        def infllm_window_forward(self, args, stream):
            a = dict(zip(fields, _sink_window._ARGS.unpack(args)))
            n = B * a["n_q"] * H * D
            rooms.append(torch.empty((n + 16,), dtype=torch.bfloat16, device="cuda"))
            rooms[-1][off:off + n] = now[0].flatten()
            assert a["d_q"] % 16 == 0 and a["q_sl"] == H * D and rooms[-1].data_ptr() % 16 == 0
            a["d_q"] = rooms[-1].data_ptr() + 2 * off
            return lib.infllm_window_forward(_sink_window._ARGS.pack(*(a[f] for f in fields)), stream)
    now = [None]

    def run():
        past, outs, at = None, [], 0
        for n in calls:
            now[0], k, v = (t[:, at:at + n].contiguous() for t in x)
            o, past = forward(None, now[0], k, rope, True, past, same, same, lambda _: v, same, D, H, Hkv)
            outs.append(o)
            at += n
        return torch.cat(outs, dim=1).float()
    want = run()
    monkeypatch.setattr(_sink_window._lib, "load", lambda: Moved())
    got = run()
    assert len(rooms) == len(calls)
    # (as above: roundings of rotated elements, probabilities and results to bf16)
    assert torch.equal(got, want) if off == 8 else float((got - want).norm()) <= 2.0 ** -7 * float(want.norm())
