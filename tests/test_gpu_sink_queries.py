"""Queries that the attention rotates to the sinks' angle itself: more sinks than a key split has tiles (splits that begin among the
sinks, that cross into them, that see none), calls that are no whole tile of queries, rows of the projection apart or next to each
other - the same bits either way, and oracle.siblings' results (2e-2 / 2e-3, the bounds of the other tests of these types)."""
import pytest
import torch

from oracle.rope import RopeOracle
from oracle.siblings import SinkWindowOracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["stream-llm", "infinite-lm"])
@pytest.mark.parametrize("D,H,Hkv,B", [(128, 4, 2, 1), (64, 6, 3, 2), (128, 5, 1, 2), (64, 4, 4, 1)])
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
