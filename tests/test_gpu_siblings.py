"""The sink + window attention types and plain causal attention on the GPU, through the attention-type registry,
against oracle.siblings on the same bf16-rounded inputs (max-abs 2e-2 / mean-abs 2e-3)."""
import pytest
import torch

from oracle.rope import RopeOracle
from oracle.siblings import CausalOracle, SinkWindowOracle

pytestmark = pytest.mark.gpu

D, MAX_ABS, MEAN_ABS = 128, 2e-2, 2e-3


def _stream(T, H, Hkv, seed, B=1):
    g = torch.Generator().manual_seed(seed)
    mk = lambda h: torch.randn(B, T, h * D, generator=g).bfloat16()
    return mk(H), mk(Hkv), mk(Hkv)


def _drive(forward, x_q, x_k, x_v, calls, H, Hkv, base):
    """Call the attention type the way a patched decoder layer does, with identity projections."""
    from infllm_amd.attention import RotaryEmbeddingESM
    rope = RotaryEmbeddingESM(D, base=base, device="cuda")
    xq, xk, xv = x_q.cuda(), x_k.cuda(), x_v.cuda()
    past, outs, pos = None, [], 0
    for L in calls:
        sl = slice(pos, pos + L)
        kv = torch.cat((xk[:, sl], xv[:, sl]), dim=-1)
        o, past = forward(None, xq[:, sl], kv, rope, True, past, lambda t: t, lambda t: t[..., :Hkv * D], lambda t: t[..., Hkv * D:],
                          lambda t: t, D, H, Hkv)
        outs.append(o)
        pos += L
    torch.cuda.synchronize()
    return torch.cat(outs, dim=1).cpu(), past


def _heads(x, h):
    B, T, _ = x.shape
    return x.view(B, T, h, D).permute(0, 2, 1, 3).float()


def _check(got, want):
    B, H, T, _ = want.shape
    err = (got.float().view(B, T, H, D).permute(0, 2, 1, 3) - want).abs()
    assert float(err.max()) <= MAX_ABS and float(err.mean()) <= MEAN_ABS, (float(err.max()), float(err.mean()))


@pytest.mark.parametrize("kind", ["stream-llm", "infinite-lm"])
@pytest.mark.parametrize("calls,n_local,n_init", [([700], 256, 16), ([300, 1, 1, 1, 250, 47], 128, 8), ([1] * 40 + [90], 64, 4),
                                                  ([5, 200], 96, 0), ([150], 256, 16)])
def test_sink_window_types_follow_oracle(kind, calls, n_local, n_init):
    from infllm_amd.attention import ATTN_FORWRAD
    H, Hkv, T = 4, 2, sum(calls)
    xq, xk, xv = _stream(T, H, Hkv, seed=T + n_init, B=2)
    got, past = _drive(ATTN_FORWRAD[kind](n_local, n_init, fattn=False), xq, xk, xv, calls, H, Hkv, 1e4)
    ora = SinkWindowOracle(RopeOracle(D, base=1e4), n_local, n_init, kind)
    want, pos = [], 0
    for L in calls:
        sl = slice(pos, pos + L)
        want.append(ora.append(_heads(xq[:, sl], H), _heads(xk[:, sl], Hkv), _heads(xv[:, sl], Hkv)))
        pos += L
    _check(got, torch.cat(want, dim=2))
    assert past[2] == T and past[0].shape[2] == min(T, n_local + n_init) == past[1].shape[2]     # stream_llm.py:43-52


@pytest.mark.parametrize("kind", ["stream-llm", "infinite-lm", "origin"])
def test_sibling_types_with_heads_of_64(kind, monkeypatch):
    """head_dim 64 through the same three types, in rows of their own width."""
    import sys
    from infllm_amd.attention import ATTN_FORWRAD
    monkeypatch.setattr(sys.modules[__name__], "D", 64)
    H, Hkv, calls, n_local, n_init = 4, 2, [300, 1, 1, 250], 128, 8
    T = sum(calls)
    xq, xk, xv = _stream(T, H, Hkv, seed=17, B=2)
    fwd = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](n_local, n_init, fattn=False)
    got, past = _drive(fwd, xq, xk, xv, calls, H, Hkv, 1e4)
    ora = CausalOracle(RopeOracle(64, base=1e4)) if kind == "origin" else SinkWindowOracle(RopeOracle(64, base=1e4), n_local, n_init, kind)
    want, pos = [], 0
    for L in calls:
        sl = slice(pos, pos + L)
        want.append(ora.append(_heads(xq[:, sl], H), _heads(xk[:, sl], Hkv), _heads(xv[:, sl], Hkv)))
        pos += L
    _check(got, torch.cat(want, dim=2))
    assert past[0].shape[-1] == 64


def test_origin_type_is_causal_attention():
    from infllm_amd.attention import ATTN_FORWRAD
    H, Hkv, calls = 4, 4, [200, 1, 1, 130]
    T = sum(calls)
    xq, xk, xv = _stream(T, H, Hkv, seed=3)
    got, past = _drive(ATTN_FORWRAD["origin"](False), xq, xk, xv, calls, H, Hkv, 5e5)
    ora = CausalOracle(RopeOracle(D, base=5e5))
    want, pos = [], 0
    for L in calls:
        sl = slice(pos, pos + L)
        want.append(ora.append(_heads(xq[:, sl], H), _heads(xk[:, sl], Hkv), _heads(xv[:, sl], Hkv)))
        pos += L
    _check(got, torch.cat(want, dim=2))
    assert past[0].shape[2] == T


@pytest.mark.parametrize("pos0,consecutive", [(0, True), (777, True), (4095, False), (1000003, True)])
def test_rope_rows_matches_fp64_rotation(pos0, consecutive):
    from infllm_amd import ops
    B, H, L = 2, 3, 37
    g = torch.Generator().manual_seed(pos0 % 97)
    full = torch.randn(B, L + 5, H * D, generator=g).bfloat16()
    x = full.cuda()[:, 2:2 + L].view(B, L, H, D).permute(0, 2, 1, 3)          # strided rows, as the forwards pass them
    rope = RopeOracle(D, base=1e6)
    got = ops.rope_rows(x, rope.inv_freq.float().cuda(), 1.0, pos0, consecutive).cpu().double()
    xf = full[:, 2:2 + L].view(B, L, H, D).permute(0, 2, 1, 3).double()
    pos = torch.arange(L, dtype=torch.float64) * (1 if consecutive else 0) + pos0
    ang = pos[:, None] * rope.inv_freq.double()[None, :]
    lo, hi = xf[..., :D // 2], xf[..., D // 2:]
    want = torch.cat((lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin()), dim=-1)
    assert float((got - want).abs().max()) <= 2 ** -7 * float(want.abs().max())      # one bf16 rounding
    empty = ops.rope_rows(x[:, :, :0], rope.inv_freq.float().cuda(), 1.0, 0)
    assert empty.shape == (B, H, 0, D)


@pytest.mark.parametrize("kind,T,H,Hkv", [("origin", 1500, 32, 8), ("origin", 2048, 32, 8), ("origin", 705, 12, 4), ("infinite-lm", 1100, 32, 8)])
def test_key_splits_of_a_prompts_first_call_follow_the_oracle(kind, T, H, Hkv):
    """A prompt whose longest rows decide how many key splits its first call is cut into (bounds of this file: bf16 outputs)."""
    from infllm_amd.attention import ATTN_FORWRAD
    xq, xk, xv = _stream(T, H, Hkv, seed=T)
    heads = _heads(xq, H), _heads(xk, Hkv), _heads(xv, Hkv)
    if kind == "origin":
        got, _ = _drive(ATTN_FORWRAD[kind](False), xq, xk, xv, [T], H, Hkv, 1e4)
        want = CausalOracle(RopeOracle(D, base=1e4)).append(*heads)
    else:
        got, _ = _drive(ATTN_FORWRAD[kind](1024, 64, fattn=False), xq, xk, xv, [T], H, Hkv, 1e4)
        want = SinkWindowOracle(RopeOracle(D, base=1e4), 1024, 64, kind).append(*heads)
    _check(got, want)


# ---- a cache that grows in place: its tensors are the filled part of buffers that the next call writes on
N_LOCAL, N_INIT = 700, 16          # every stream below stays inside: nothing is cut


class _Branch:
    """A stream of one of the types, fed [batch, tokens, heads * D] rows, with the oracle following it."""

    def __init__(self, kind, H, Hkv, past=None, history=()):
        from infllm_amd.attention import ATTN_FORWRAD
        self.kind, self.H, self.Hkv, self.past, self.history = kind, H, Hkv, past, list(history)
        self.forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](N_LOCAL, N_INIT, fattn=False)

    def feed(self, rows):
        from infllm_amd.attention import RotaryEmbeddingESM
        q, k, v = (t.cuda() for t in rows)
        same = lambda t: t
        o, self.past = self.forward(None, q, k, RotaryEmbeddingESM(D, base=1e4, device="cuda"), True, self.past, same, same, lambda _: v, same, D, self.H,
                                    self.Hkv)
        self.history.append(rows)
        return o

    def check(self, o):
        """the last call's rows against the oracle over the whole history (bounds of this file)"""
        rope = RopeOracle(D, base=1e4)
        ora = CausalOracle(rope) if self.kind == "origin" else SinkWindowOracle(rope, N_LOCAL, N_INIT, self.kind)
        for q, k, v in self.history:
            want = ora.append(_heads(q, self.H), _heads(k, self.Hkv), _heads(v, self.Hkv))
        _check(o.cpu(), want)

    def fork(self, past=None, history=None):
        return _Branch(self.kind, self.H, self.Hkv, self.past if past is None else past, self.history if history is None else history)

    def cut(self, change):
        """the cache with `change` made to its tensors"""
        return tuple(change(t) if torch.is_tensor(t) else t for t in self.past)


KINDS = ["origin", "stream-llm", "infinite-lm"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("B", [1, 2])
def test_two_continuations_of_one_prompt(kind, B):
    """The first one goes on in the prompt's buffers, the second finds them taken and copies; neither sees the other's rows."""
    H, Hkv = 4, 2
    prompt = _Branch(kind, H, Hkv)
    prompt.check(prompt.feed(_stream(300, H, Hkv, 1, B)))
    kept = [t.clone() for t in prompt.past[:2]]
    a, b = prompt.fork(), prompt.fork()
    for i, n in enumerate([1, 1, 40, 1]):
        a.check(a.feed(_stream(n, H, Hkv, 10 + i, B)))
        if i == 0:
            assert a.past[0].data_ptr() == prompt.past[0].data_ptr()
        b.check(b.feed(_stream(n, H, Hkv, 20 + i, B)))
        assert a.past[0].data_ptr() != b.past[0].data_ptr() and a.past[0].shape == b.past[0].shape
    again = prompt.fork()
    again.check(again.feed(_stream(7, H, Hkv, 30, B)))
    assert all(torch.equal(x, y) for x, y in zip(kept, prompt.past[:2]))


@pytest.mark.parametrize("kind", KINDS)
def test_changed_caches_continue_in_buffers_of_their_own(kind):
    """rolled back by some tokens, rows of the batch in another order, one prompt for a whole batch, one row of the batch"""
    H, Hkv, B = 4, 2, 2
    base = _Branch(kind, H, Hkv)
    base.feed(_stream(300, H, Hkv, 1, B))
    rows = base.history[0]
    kept = [t.clone() for t in base.past[:2]]
    seen = lambda past, n: past if kind == "origin" else (past[0], past[1], n, past[3])
    back = base.fork(seen(tuple(t[:, :, :280] if torch.is_tensor(t) and t.shape[2] == 300 else t for t in base.past), 280), [tuple(t[:, :280] for t in rows)])
    order = base.fork(base.cut(lambda t: t[[1, 0]]), [tuple(t[[1, 0]] for t in rows)])
    one = base.fork(base.cut(lambda t: t[1:]), [tuple(t[1:] for t in rows)])
    many = base.fork(base.cut(lambda t: t[:1].expand(3, -1, -1, -1)), [tuple(t[:1].expand(3, -1, -1) for t in rows)])
    for i, (branch, batch) in enumerate(((back, B), (order, B), (one, 1), (many, 3))):
        for n in (1, 30, 1):
            branch.check(branch.feed(_stream(n, H, Hkv, 40 + 3 * i + n, batch)))
        assert branch.past[0].data_ptr() != base.past[0].data_ptr()
    assert all(torch.equal(x, y) for x, y in zip(kept, base.past[:2]))
    base.check(base.feed(_stream(1, H, Hkv, 60, B)))


@pytest.mark.parametrize("kind", KINDS)
def test_growth_past_the_room(kind):
    """200 tokens leave room for 256 more; the calls cross its end by one token, exactly, and by many"""
    H, Hkv = 4, 2
    for calls in ([200, 255, 1, 1], [200, 256, 1], [200, 250, 20, 1], [200, 1, 400]):
        s = _Branch(kind, H, Hkv)
        for i, n in enumerate(calls):
            o = s.feed(_stream(n, H, Hkv, 70 + i))
        s.check(o)
        assert s.past[0].shape[2] == sum(calls)


def test_a_dropped_cache_is_given_back():
    H, Hkv = 4, 2
    rows = _stream(300, H, Hkv, 1), _stream(1, H, Hkv, 2)
    s = _Branch("origin", H, Hkv)
    s.feed(rows[0])
    del s
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    s = _Branch("origin", H, Hkv)
    s.feed(rows[0])
    s.feed(rows[1])
    assert torch.cuda.memory_allocated() > before
    del s
    assert torch.cuda.memory_allocated() == before
