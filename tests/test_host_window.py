"""CPU-only checks of the sliding-window and causal attention types' host side: what reaches the native call, with a stand-in
for the library that records it."""
import threading
import weakref

import pytest
import torch

from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM, _sink_window

H, HKV, D, B = 4, 2, 128, 2


class Native:
    """records the argument blocks of infllm_window_forward instead of launching"""

    def __init__(self):
        self.calls = []

    def infllm_window_forward(self, args, stream):
        self.calls.append((_sink_window._ARGS.unpack(args), stream))
        return 0


@pytest.fixture
def native(monkeypatch):
    lib = Native()
    monkeypatch.setattr(_sink_window._lib, "load", lambda: lib)
    monkeypatch.setattr(_sink_window, "_stream", lambda: 7)
    monkeypatch.setattr(_sink_window, "_on_gpu", lambda t: True)
    return lib


def layer(kind, past, n, batch=B, q=None, k=None, v=None):
    fwd = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](64, 8, fattn=False)
    same = lambda t: t
    rows = lambda h: torch.zeros((batch, n, h * D), dtype=torch.bfloat16)
    q, k, v = rows(H) if q is None else q, rows(HKV) if k is None else k, rows(HKV) if v is None else v
    return fwd(None, torch.zeros((batch, n, 1)), torch.zeros((batch, n, 1)), RotaryEmbeddingESM(D, device="cpu"), True, past, lambda _: q, lambda _: k,
               lambda _: v, same, D, H, HKV)


KINDS = ["origin", "stream-llm", "infinite-lm"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("what", ["batch", "heads", "width", "dtype", "device", "rank", "short values", "values' batch"])
def test_a_cache_that_does_not_fit_the_call_is_refused(kind, what, native):
    """(the native call would read, and copy, rows beyond the end of such a cache)"""
    _, past = layer(kind, None, 30)
    k, v, rest = past[0], past[1], past[2:]
    bad = {"batch": lambda t: t[:1], "heads": lambda t: t[:, :1], "width": lambda t: t[..., :64], "dtype": lambda t: t.half(),
           "device": lambda t: t.to("meta"), "rank": lambda t: t[0], "short values": lambda t: t[:, :, :20], "values' batch": lambda t: t[:1]}[what]
    if what not in ("short values", "values' batch"):
        k = bad(k)
    v = bad(v)
    n = len(native.calls)
    with pytest.raises((ValueError, IndexError)):
        layer(kind, (k, v) + tuple(rest), 1)
    assert len(native.calls) == n


def test_un_rotated_sinks_that_do_not_fit_the_call_are_refused(native):
    _, past = layer("infinite-lm", None, 30)
    for bad in (past[3][:1], past[3][:, :1], past[3].float(), past[3].to("meta")):
        with pytest.raises(ValueError):
            layer("infinite-lm", past[:3] + (bad,), 1)
    assert len(native.calls) == 1


@pytest.mark.parametrize("kind", KINDS)
def test_projections_of_another_length_or_batch_are_refused(kind, native):
    rows = lambda b, n, h: torch.zeros((b, n, h * D), dtype=torch.bfloat16)
    for bad in (dict(q=rows(B, 29, H)), dict(k=rows(B - 1, 30, HKV)), dict(v=rows(B, 31, HKV)), dict(v=rows(B, 30, HKV).to("meta"))):
        with pytest.raises((RuntimeError, ValueError)):
            layer(kind, None, 30, **bad)
    assert not native.calls
    layer(kind, None, 30, q=rows(B, 30, H).view(B * 30, H * D), k=rows(B, 30, HKV).view(B, 30, HKV, D))    # other shapes of the same rows are taken
    assert len(native.calls) == 1


@pytest.mark.parametrize("kind", KINDS)
def test_a_cache_that_fits_is_taken(kind, native):
    _, past = layer(kind, None, 30)
    for n in (1, 20, 60, 1):
        out, past = layer(kind, past, n)
        assert out.shape == (B, n, H * D)
    assert len(native.calls) == 5 and past[0].shape == past[1].shape


@pytest.mark.parametrize("kind", KINDS)
def test_a_cache_can_be_copied_pickled_and_saved(kind, native):
    """Keeping a prompt's cache for later continuations is a normal use; the copies are caches of their own."""
    import copy
    import io
    import pickle
    _, past = layer(kind, None, 30)
    for t in past[:2]:
        t.normal_()
    saved = io.BytesIO()
    torch.save(past, saved)
    saved.seek(0)
    for other in (copy.deepcopy(past), pickle.loads(pickle.dumps(past)), torch.load(saved, weights_only=True), tuple(copy.copy(past))):
        assert all(torch.equal(a, b) for a, b in zip(other[:2], past[:2]))
        _, new = layer(kind, other, 1)
        if other[0].data_ptr() != past[0].data_ptr():
            assert new[0].data_ptr() not in (other[0].data_ptr(), past[0].data_ptr())
    assert past[0].shape[2] == 30


def test_a_call_on_another_stream_gets_buffers_of_its_own(native, monkeypatch):
    """Buffers belong to the stream they were allocated on: the allocator may hand them out again in that stream's order while
    another stream still writes them."""
    _, past = layer("origin", None, 30)
    _, same = layer("origin", past, 1)
    assert same[0].data_ptr() == past[0].data_ptr()
    monkeypatch.setattr(_sink_window, "_stream", lambda: 8)
    _, other = layer("origin", same, 1)
    assert other[0].data_ptr() != same[0].data_ptr() and other[1].data_ptr() != same[1].data_ptr() and native.calls[-1][1] == 8
    _, again = layer("origin", other, 1)
    assert again[0].data_ptr() == other[0].data_ptr()


def test_which_calls_write_behind_the_cache_they_are_given(native):
    """Only a continuation of the newest cache of the buffers, unchanged, with room behind it; every other call copies."""
    _, p = layer("origin", None, 30)                                                  # room for 256 more
    where = lambda past: (past[0].data_ptr(), past[1].data_ptr())
    _, a = layer("origin", p, 1)
    _, b = layer("origin", p, 1)
    assert where(a) == where(p) and where(b) != where(p)
    for other in ((b[0][:, :, :30], b[1][:, :, :30]), (b[0][[1, 0]], b[1][[1, 0]]), (b[0], a[1]), (a[0], b[1]), (b[1], b[0]),
                  (b[0][:1].expand(B, -1, -1, -1), b[1][:1].expand(B, -1, -1, -1))):
        _, c = layer("origin", other, 1)
        assert where(c)[0] not in (where(a)[0], where(b)[0]) and where(c)[1] not in (where(a)[1], where(b)[1])
    _, full = layer("origin", b, 256)                                                 # exactly to the end
    assert where(full) == where(b)
    _, beyond = layer("origin", full, 1)
    assert where(beyond) != where(full) and beyond[0].shape[2] == 288
    _, same = layer("origin", (beyond[0].detach(), beyond[1].detach()), 1)            # another tensor of the same rows
    assert where(same) == where(beyond)


def tickets(native):
    names = [n for n, _ in _sink_window._lib.WindowArgs._fields_]
    return [args[names.index("d_ticket")] for args, _ in native.calls]


@pytest.mark.parametrize("kind", KINDS)
def test_a_captured_step_keeps_no_address_of_shared_words(kind, native, monkeypatch):
    """A graph may be replayed beside another that was captured on the same stream, beside eager steps, and long after: its steps
    count in words of their own scratch, also where a warm-up has made words already."""
    _, past = layer(kind, None, 30)
    _, past = layer(kind, past, 1)
    assert tickets(native)[-1] != 0
    monkeypatch.setattr(_sink_window, "_capturing", lambda dev: True, raising=False)
    _, past = layer(kind, past, 1)
    assert tickets(native)[-1] == 0
    layer(kind, past, 1)
    assert tickets(native)[-1] == 0


class Words:
    """remembers which tensors of 32-bit words torch.zeros and torch.empty have made, and whether they are still there"""

    def __init__(self, monkeypatch, before=lambda: None):
        self.made = []

        def remembering(make):
            def call(shape, **kw):
                if kw.get("dtype") is not torch.int32:
                    return make(shape, **kw)
                before()
                t = make(shape, **kw)
                self.made.append((t.data_ptr(), t.numel() * 4, weakref.ref(t)))
                return t
            return call
        for name in ("zeros", "empty"):
            monkeypatch.setattr(torch, name, remembering(getattr(torch, name)))

    def owner(self, address, words):
        """the tensor that is alive and holds the words at that address"""
        return [r for at, size, r in self.made if r() is not None and at <= address and address + 4 * words <= at + size]


@pytest.mark.parametrize("kind", KINDS)
def test_two_threads_steps_count_in_words_that_stay(kind, native, monkeypatch):
    """Both make words at once, for one stream: whichever are kept, the kernels got addresses of memory that is not given away."""
    meet = threading.Barrier(2)
    words = Words(monkeypatch, lambda: meet.wait(timeout=20))
    caches = [None, None]

    def step(i):
        caches[i] = layer(kind, None, 1)[1]
    threads = [threading.Thread(target=step, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(native.calls) == 2 and all(caches)
    for address in tickets(native):
        assert words.owner(address, B * H)


@pytest.mark.parametrize("kind", KINDS)
def test_words_of_a_cache_are_used_by_one_call_at_a_time(kind, native, monkeypatch):
    """A second continuation of a prompt, which another thread or another stream may make, has words of its own; so has a larger
    batch; and none are replaced while a launch may count in them.  Words that hold anything yet are said to."""
    words = Words(monkeypatch)
    _, prompt = layer(kind, None, 70)
    inside = {}
    launch = native.infllm_window_forward

    def meanwhile(args, stream):                              # a step within the step: as two threads do it
        status = launch(args, stream)
        if not inside:
            inside["cache"] = None
            inside["cache"] = layer(kind, prompt, 1)[1]
        return status
    monkeypatch.setattr(native, "infllm_window_forward", meanwhile)
    _, one = layer(kind, prompt, 1)
    first, second = tickets(native)[-2:]
    assert first and second and first != second
    assert words.owner(first, B * H) and words.owner(second, B * H)
    _, one = layer(kind, one, 1)
    assert tickets(native)[-1] in (first, second)             # (a cache's steps go on with its words)
    _, large = layer(kind, None, 1, batch=400)
    assert words.owner(tickets(native)[-1], 400 * H) and tickets(native)[-1] not in (first, second)
    assert words.owner(first, B * H) or words.owner(second, B * H)
    monkeypatch.setattr(_sink_window, "_stream", lambda: 8)
    _, other = layer(kind, one, 1)
    assert tickets(native)[-1] not in (0, first, second)      # (two streams' launches have no order)
    layer(kind, other, 1)
    assert [args[-1] for args, _ in native.calls] == [1, 0, 1, 0, 1, 1, 0]


def test_a_step_takes_no_more_scratch_than_its_cache_brings(native, monkeypatch):
    """A causal cache of 248 query rows of 128 keeps a step's scratch of just under 4 MiB; a step of the sink + window types over the same
    cache has the queries twice and takes more than is kept."""
    made = []

    def remembering(make):
        def call(*args, **kw):
            t = make(*args, **kw)
            made.append((t.data_ptr(), t.numel() * t.element_size(), weakref.ref(t)))
            return t
        return call
    monkeypatch.setattr(torch, "empty", remembering(torch.empty))
    fields = [n for n, _ in _sink_window._lib.WindowArgs._fields_]
    inside = []

    def launch(args, stream):                                 # (while the call holds what it made)
        a = dict(zip(fields, _sink_window._ARGS.unpack(args)))
        inside.append(any(r() is not None and at <= a["d_work"] and a["d_work"] + a["work_bytes"] <= at + size for at, size, r in made))
        return 0
    monkeypatch.setattr(native, "infllm_window_forward", launch)
    _, past = layer("origin", None, 30, batch=62)
    _, past = layer("origin", past, 1, batch=62)
    for kind in ("stream-llm", "origin"):
        _, more = layer(kind, past if kind == "origin" else (past[0], past[1], 31, None), 1, batch=62)
    layer("stream-llm", (more[0], more[1], 32, None), 1, batch=62)
    assert inside == [True] * 5


def misaligned(*shape):
    """contiguous, but two bytes off"""
    n = 1
    for d in shape:
        n *= d
    return torch.arange(n + 8).bfloat16()[1:1 + n].view(shape)


def test_rows_are_handed_on_aligned():
    """(contiguous() gives a contiguous tensor back however it is aligned, and whatever the strides of its single-element dims)"""
    from infllm_amd.ops import rows16
    single = torch.zeros((1, 2, 1, 128), dtype=torch.bfloat16).as_strided((1, 2, 1, 128), (3, 128, 5, 1))
    odd = torch.zeros((2, 3, 5, 130), dtype=torch.bfloat16)[..., :128]
    for t in (misaligned(2, 3, 5, 128), single, odd, torch.zeros((2, 3, 128, 5), dtype=torch.bfloat16).transpose(2, 3)):
        r = rows16(t)
        assert torch.equal(r, t) and r.data_ptr() % 16 == 0 and r.stride(3) == 1 and all(s % 8 == 0 for s in r.stride()[:3])
    fine = torch.zeros((2, 5, 3, 128), dtype=torch.bfloat16).transpose(1, 2)
    assert rows16(fine) is fine


@pytest.mark.parametrize("kind", KINDS)
def test_misaligned_rows_and_caches_are_copied(kind, native):
    _, past = layer(kind, None, 30)
    cache = tuple(misaligned(*t.shape) if torch.is_tensor(t) else t for t in past)
    layer(kind, cache, 1, q=misaligned(B, 1, H * D), k=misaligned(B, 1, HKV * D), v=misaligned(B, 1, HKV * D))
    fields = [n for n, _ in _sink_window._lib.WindowArgs._fields_]
    args = dict(zip(fields, native.calls[-1][0]))
    addresses = {n: args[n] for n in fields if n.startswith("d_") and n != "d_inv_freq"}
    assert addresses["d_old_k"] and all(a % 16 == 0 for a in addresses.values()), addresses
