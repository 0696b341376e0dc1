"""Inputs that are no numbers: a NaN or an infinity reaches the rows that read it, as in the softmax of the oracle, and no others.
(Numbers are compared by the bounds of the other tests: bf16 outputs, max-abs 2e-2.)"""
import pytest
import torch

from oracle.multistage import MultiStageOracle
from oracle.rope import RopeOracle
from oracle.siblings import CausalOracle, SinkWindowOracle
from stream_parity import SMALL, feed, make_stream, new_manager

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def same_kind(got, want):
    got, want = got.float().cpu(), want.float().cpu()
    nan = got.isnan(), want.isnan()
    assert bool((nan[0] == nan[1]).all()), [int(n.sum()) for n in nan]
    ok = want.isfinite()
    assert bool((got == want)[~ok & ~nan[1]].all()), "infinities"
    assert not ok.any() or float((got[ok] - want[ok]).abs().max()) <= 2e-2


POISON = {
    "one key": lambda q, k, v: k[0, 0, 100:101, 3].fill_(NAN),
    "four keys of a lane": lambda q, k, v: k[0, 0, 96:100].fill_(NAN),
    "a split's keys": lambda q, k, v: k[0, 0, 128:256].fill_(NAN),
    "every key of a head": lambda q, k, v: k[0, 0].fill_(NAN),
    "an infinite key": lambda q, k, v: k[0, 0, 100, 3].fill_(INF),                 # its logit: + or - infinity by the query's sign
    "the last key": lambda q, k, v: k[0, 0, -1, 3].fill_(-INF),
    "one query": lambda q, k, v: q[0, 1, -1, 5].fill_(NAN),
    "a value": lambda q, k, v: v[0, 0, 100, 3].fill_(NAN),
    "an infinite value": lambda q, k, v: v[0, 0, 100, 3].fill_(-INF),
    "the last value": lambda q, k, v: v[0, 0, -1, 3].fill_(INF),
}


@pytest.mark.parametrize("what", POISON)
@pytest.mark.parametrize("Lq", [1, 40])
@pytest.mark.parametrize("G", [1, 2, 4])
def test_operator(what, Lq, G):
    from infllm_amd.attention.dot_production_attention import get_multi_stage_dot_production_attention
    Hkv, H, n1, n2 = 2, 2 * G, 589, 70
    g = torch.Generator().manual_seed(G)
    mk = lambda h, n: torch.randn(1, h, n, 128, generator=g).bfloat16()
    q, k, v, k2, v2 = mk(H, Lq), mk(Hkv, n1), mk(Hkv, n1), mk(Hkv, n2), mk(Hkv, n2)
    POISON[what](q, k, v)
    Attn, _ = get_multi_stage_dot_production_attention(False)
    attn, ora = Attn(q.shape, torch.bfloat16, "cuda"), MultiStageOracle(q.shape)
    for a, dev in ((attn, lambda t: t.cuda()), (ora, lambda t: t.float())):
        a.append(dev(q), dev(k), dev(v), sliding_window=1000)
        a.append(dev(q), dev(k2), dev(v2), end=True)
    same_kind(attn.get_result()[0], ora.get_result()[0])


# (an infinite component rotates into two, whose signs depend on where positions are counted from: for the types with a window
# the oracle counts from the window's start, so only the causal type's logit is the oracle's infinity)
@pytest.mark.parametrize("what,kind", [(w, t) for w in POISON for t in ("origin", "stream-llm", "infinite-lm")
                                       if t == "origin" or w not in ("an infinite key", "the last key")])
@pytest.mark.parametrize("dim", [128, 64])
def test_one_token_of_the_window_types(what, kind, dim):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    H, Hkv, n, n_local, n_init = 4, 2, 333, 300, 8                     # a token behind them: the sinks have left the window
    g = torch.Generator().manual_seed(dim)
    q, k, v = (torch.randn(1, h, n + 1, dim, generator=g).bfloat16() for h in (H, Hkv, Hkv))
    POISON[what](q, k[:, :, :n] if "last" not in what else k, v[:, :, :n] if "last" not in what else v)
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](n_local, n_init, fattn=False)
    rope = RopeOracle(dim, base=1e4)
    ora = CausalOracle(rope) if kind == "origin" else SinkWindowOracle(rope, n_local, n_init, kind)
    past, same = None, lambda t: t
    rows = lambda t, a, b: t[:, :, a:b].transpose(1, 2).reshape(1, b - a, -1).cuda()
    for a, b in ((0, n), (n, n + 1)):
        got, past = forward(None, rows(q, a, b), rows(k, a, b), RotaryEmbeddingESM(dim, base=1e4, device="cuda"), True, past, same, same,
                            lambda _: rows(v, a, b), same, dim, H, Hkv)
        want = ora.append(q[:, :, a:b].float(), k[:, :, a:b].float(), v[:, :, a:b].float())
    same_kind(got.view(1, 1, H, dim).transpose(1, 2), want)


@pytest.mark.parametrize("driven", ["resident", "host"])
@pytest.mark.parametrize("what", ["key", "value", "query"])
def test_one_token_of_the_streaming_memory(what, driven, monkeypatch):
    """A NaN of one head in the window (or in the token's query): that head's rows become NaN, the others stay as they are."""
    from infllm_amd.attention import ContextManager
    if driven == "host":
        monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    H, Hkv, T = 8, 2, 705
    q, k, v = (t.cuda() for t in make_stream(T, H, Hkv, 3))
    clean = feed(new_manager(1e4, **SMALL), q, k, v, [700, 1, 1, 1, 1, 1])[-2:]
    hit = range(2, 3) if what == "query" else range(4)                 # the poisoned head, or the query heads of kv head 0
    if what == "query":
        q[:, 2, 703:, 7] = NAN
    else:
        (k if what == "key" else v)[:, 0, 701, 7] = NAN
    got = feed(new_manager(1e4, **SMALL), q, k, v, [700, 1, 1, 1, 1, 1])[-2:]
    for a, b in zip(got, clean):
        if what == "value":
            assert a[:, hit, :, 7].isnan().all()
            a[:, hit, :, 7] = b[:, hit, :, 7]
            assert torch.equal(a, b)
            continue
        keep = [h for h in range(H) if h not in hit]
        assert a[:, hit].isnan().all() and a[:, keep].isfinite().all()
        if what == "key":                                              # (a NaN in a query also moves the selection, made by a mean over all heads)
            assert torch.equal(a[:, keep], b[:, keep])
