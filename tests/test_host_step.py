"""A step that csrc/host.cpp makes is the step of the general way in _sink_window.py: the same argument block - sizes, strides, places, which
addresses are there and which of them are the same - and a cache of the same sizes, over first steps, caches that grow, fill and are
cut, sinks that are still being collected, rows and caches out of the ordinary, continuations of an older cache."""
import types

import pytest
import torch

from infllm_amd import _lib
from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM, _sink_window

FIELDS = [n for n, _ in _lib.WindowArgs._fields_]


def odd(t):
    """the same rows, two bytes off"""
    flat = torch.zeros(t.numel() + 8, dtype=t.dtype)
    return flat[1:1 + t.numel()].view(t.shape).copy_(t)


def schedule(kind, H, HKV, D, B, plain, monkeypatch):
    real, calls, steps = _lib.host(), [], []

    def forward(args, stream):
        a = dict(zip(FIELDS, _sink_window._ARGS.unpack(args)))
        at = {n: a.pop(n) for n in FIELDS if n.startswith("d_")}
        calls.append((stream, a, {n: bool(p) for n, p in at.items()}, at["d_cache_k"] == at["d_old_k"], at["d_cache_v"] == at["d_old_v"],
                      at["d_raw"] == at["d_raw_old"], at["d_inv_freq"]))
        return 0

    def step(*args):
        got = real.step(*args) if plain else None
        steps.append(got is not None)
        return got
    native = types.SimpleNamespace(infllm_window_forward=forward)
    monkeypatch.setattr(_lib, "load", lambda: native)
    monkeypatch.setattr(_lib, "host", lambda: types.SimpleNamespace(step=step, claim=real.claim, make_room=real.make_room))
    monkeypatch.setattr(_sink_window, "_stream", lambda: 0)
    monkeypatch.setattr(_sink_window, "_on_gpu", lambda t: True)
    fwd = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](40, 8, fattn=False)
    same, seen = (lambda t: t), []

    def call(past, n, rows=lambda t: t):
        q, k, v = (rows(torch.zeros((B, n, h * D), dtype=torch.bfloat16)) for h in (H, HKV, HKV))
        hidden = torch.zeros((B, n, 1))
        out, past = fwd(None, hidden, hidden, ROPE[D], True, past, lambda _: q, lambda _: k, lambda _: v, same, D, H, HKV)
        seen.append((out.shape, out.stride(), past[0].shape, past[0].stride(), past[1].stride(), past[2:3], None if len(past) < 4 or past[3] is None else past[3].shape))
        return past
    past = None
    for n in (1, 1, 3, 1, 1, 1, 1):                       # from nothing, the sinks one by one
        past = call(past, n)
    older = past
    for _ in range(45):                                   # over the edge where a cache with a window is cut
        past = call(past, 1)
    call(older, 1)                                        # a second continuation
    past = call(past, 1, odd)
    past = call(past, 1, lambda t: torch.cat((t, t), dim=1)[:, :1])          # rows that lie apart
    past = call(past, 1, lambda t: t.view(B, -1))
    past = call((odd(past[0]), past[1]) + past[2:], 1)
    past = call(tuple(t.clone() if torch.is_tensor(t) else t for t in past), 1)
    call(call(past, 5), 1)
    past = call(None, 300)
    for _ in range(3):
        past = call(past, 1)
    return calls, seen, steps


ROPE = {d: RotaryEmbeddingESM(d, device="cpu") for d in (64, 128)}


@pytest.mark.parametrize("kind", ["origin", "stream-llm", "infinite-lm"])
@pytest.mark.parametrize("H,HKV,D,B", [(4, 2, 128, 1), (6, 6, 64, 3)])
def test_a_step_is_the_general_ways(kind, H, HKV, D, B):
    with pytest.MonkeyPatch.context() as m:
        got = schedule(kind, H, HKV, D, B, True, m)
    with pytest.MonkeyPatch.context() as m:
        want = schedule(kind, H, HKV, D, B, False, m)
    assert got[0] == want[0] and got[1] == want[1]
    assert sum(got[2]) >= 45 and len(got[2]) == len(want[2])        # (the ordinary ones; the others were handed back)


def test_failures_and_other_inputs():
    host = _lib.host()
    assert host.step(*(0,) * 17) is None                            # no cache: not a plain step
    for args in ((), (1,) * 16, ("a",) * 17):
        with pytest.raises(TypeError):
            host.step(*args)
    for args in ((None, 1, 0), (torch.zeros(3), 1, 0)):
        with pytest.raises(TypeError):
            host.make_room(*args)
    with pytest.raises(TypeError):
        host.claim(None, None, 1, 0)
    t = torch.zeros((1, 2, 3, 4))
    assert host.claim(t, t, 1, 0) is None


class Other(torch.utils._python_dispatch.TorchDispatchMode):
    """runs `work` at the first view or tensor that a call makes"""
    def __init__(self, work):
        super().__init__()
        self.work = work

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        work, self.work = self.work, lambda: None
        work()
        return func(*args, **(kwargs or {}))


def plain_step(n_init, mode=None):
    """one native step behind three tokens: (what it returns, its native calls, the storage of its cache)"""
    host, H, D, calls = _lib.host(), 2, 64, []
    both = torch.zeros((2, 1, H, 8, D), dtype=torch.bfloat16)
    host.make_room(both, 3, 0)
    k, v = both.narrow(3, 0, 3).unbind(0)
    storage = k.untyped_storage()
    storage._infllm_words = (torch.zeros(64, dtype=torch.int32), 64, H, 0, 128, 1 << 20)
    rows = [torch.zeros((1, 1, H * D), dtype=torch.bfloat16) for _ in range(3)]
    args = (1, 40, n_init, *rows, (k, v, 3, None), ROPE[D].inv_freq, 1.0, 1, H, H, D, 1 << 10, 0, lambda a, s: calls.append(a) or 0, lambda words: words[1])
    with mode(storage) if mode else torch.no_grad():
        return host.step(*args), calls, storage


def test_sizes_that_the_argument_block_does_not_hold():
    assert plain_step(8)[0] is not None
    for n in (-1, 1 << 31, 1 << 40):
        got, calls, storage = plain_step(n)
        assert got is None and not calls and storage._infllm_words is not None      # (the general way refuses it)


def test_words_are_taken_before_other_code_runs():
    seen = []
    got, calls, _ = plain_step(8, lambda storage: Other(lambda: seen.append("_infllm_words" in storage.__dict__)))
    assert seen == [False] and got is not None and len(calls) == 1
