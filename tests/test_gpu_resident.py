"""Units resident in HBM (one native call per append(), selections turned into page tables on the device) against the
host-driven path, which the other stream tests hold against the oracle: the same selections, outputs and state."""
import pytest
import torch

from stream_parity import REFERENCE, SMALL, feed, make_stream, new_manager

pytestmark = pytest.mark.gpu

CASES = [
    # calls that begin inside the window, blocks that end on and off a unit, the first selection over exactly topk units, calls
    # of one token (a step) with and without a unit carved behind it
    ("small", [300, 1, 1, 700, 64, 1, 33], 8, 2, 2, dict(SMALL)),
    # calls whose blocks read nothing but the window, the last one short: merged and scored together
    ("inside the window", [200, 47, 900], 8, 2, 2, dict(SMALL, n_local=512)),
    ("fifo, tight cache", [1300, 40, 1, 500], 8, 2, 1, dict(SMALL, max_cached_block=4, cache_strategy="fifo")),
    ("steps", [420] + [1] * 70, 8, 2, 1, dict(SMALL)),
    ("no GQA, perhead", [500, 1, 200], 4, 2, 1, dict(SMALL, perhead=True)),
    ("three heads a group, no sinks", [600, 1, 130], 6, 2, 1, dict(SMALL, n_init=0)),
    ("reference", [8192, 1501, 1, 1], 32, 8, 1, dict(REFERENCE)),
    ("heads of 64", [4100, 1, 1], 12, 12, 1, dict(REFERENCE, n_local=1024, dim=64)),
    # ... the chip full of them at six key splits, scores of 32 keys a wave
    ("36 heads of 64", [3300, 700, 1], 36, 36, 1, dict(REFERENCE, n_local=1100, dim=64)),
    ("heads of 32", [900, 1, 200], 8, 2, 2, dict(SMALL, dim=32)),
]


@pytest.mark.parametrize("name,calls,H,Hkv,B,kw", CASES, ids=[c[0] for c in CASES])
def test_resident_units_give_the_host_driven_stream(name, calls, H, Hkv, B, kw, monkeypatch):
    from infllm_amd.attention import ContextManager
    T = sum(calls)
    q, k, v = (t.cuda() for t in make_stream(T, H, Hkv, 5 + T, B=B, D=kw.get("dim", 128)))
    cm = new_manager(1e4, **kw)
    got = feed(cm, q, k, v, calls)
    assert cm._resident and cm.num_global_block > kw["topk"]
    monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    ref = new_manager(1e4, **kw)
    want = feed(ref, q, k, v, calls)
    assert not ref._resident
    for n, a, b in zip(calls, got, want):
        if n > 1 and 1 not in calls[:calls.index(n)] and kw.get("dim") != 64:   # the same kernels and splits
            assert torch.equal(a, b), n
        err = (a.float() - b.float()).abs()                     # a step's splits differ
        assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, (n, float(err.max()))
    assert cm.stats == ref.stats and cm.stats["misses"] > 0
    for a, b in zip(cm.policy, ref.policy):
        assert a.cached == b.cached
    a, b = cm.export_state(), ref.export_state()
    assert a["length"] == b["length"] == T and a["n_units"] == b["n_units"] and a["init_len"] == b["init_len"]
    for name in ("tail_k", "tail_v", "init_k", "init_v"):
        assert torch.equal(a[name], b[name]), name
    assert torch.equal(a["units"], b["units"].cpu())
    assert torch.equal(a["units"][-1], cm.host_unit(cm.num_global_block - 1))
    assert torch.allclose(a["tail_score"], b["tail_score"], rtol=2e-3, atol=1e-5)


def test_leaving_and_the_budget(monkeypatch):
    """A manager whose selections are to be recorded goes over to the host-driven path in the middle of a stream, and so does
    one whose units outgrow the budget: outputs, books and slots as if the host had driven from the start."""
    import infllm_amd.attention.context_manager as manager_module
    from infllm_amd.attention import ContextManager
    from infllm_amd.attention.context_manager import _Units
    calls, kw = [700, 500, 1, 300], dict(SMALL, async_global_stream=True)
    T = sum(calls)
    q, k, v = (t.cuda() for t in make_stream(T, 8, 2, 77, B=2))
    monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    ref = new_manager(1e4, **kw)
    want = torch.cat(feed(ref, q, k, v, calls), dim=2)
    monkeypatch.setattr(ContextManager, "resident_bytes", None)
    monkeypatch.setattr(manager_module, "_UNIT_CHUNK", 8)
    before = _Units.used.get(0, 0)
    for how in ("trace", "budget"):
        cm = new_manager(1e4, **kw)
        outs = feed(cm, q, k, v, calls[:1])
        assert cm._resident and _Units.used[0] > before
        if how == "trace":
            cm.record_trace = True
        else:
            monkeypatch.setattr(ContextManager, "resident_bytes", _Units.used[0])      # the next chunk is one too many
        outs += feed(cm, q, k, v, calls[1:], pos=calls[0])
        assert cm._resident is None and _Units.used[0] == before
        assert torch.equal(torch.cat(outs, dim=2), want)
        assert cm.stats == ref.stats
        assert all(a.cached == b.cached for a, b in zip(cm.policy, ref.policy))
        monkeypatch.setattr(ContextManager, "resident_bytes", None)
        if how == "trace":
            assert len(cm.trace_blocks) == sum(-(-n // 64) for n in calls[1:])


def test_managers_of_two_threads_and_streams(monkeypatch):
    """Two threads, each with a stream and a manager of its own: workspaces, logs and the budget's books are apart or shared
    as they should be."""
    import threading
    T = 1100
    data = [tuple(t.cuda() for t in make_stream(T, 8, 2, 90 + i)) for i in range(2)]
    alone = []
    for q, k, v in data:
        alone.append(torch.cat(feed(new_manager(1e4, **SMALL), q, k, v, [700, 400]), dim=2))
    torch.cuda.synchronize()
    got = [None, None]

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            outs = []
            for _ in range(3):
                outs = feed(new_manager(1e4, **SMALL), *data[i], [700, 400])
            torch.cuda.current_stream().synchronize()
            got[i] = torch.cat(outs, dim=2)
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert torch.equal(got[0], alone[0]) and torch.equal(got[1], alone[1])


def test_managers_of_two_threads_on_one_stream():
    """Two threads on the default stream, each with a manager of its own, calls of one token and of several blocks: they share
    the calls' workspaces, and the stream orders their calls."""
    import threading
    calls = [700] + [1] * 40 + [300] + [1] * 40 + [129]
    data = [tuple(t.cuda() for t in make_stream(sum(calls), 8, 2, 190 + i)) for i in range(2)]
    alone = [torch.cat(feed(new_manager(1e4, **SMALL), *d, calls), dim=2) for d in data]
    torch.cuda.synchronize()
    got, start = [None, None], threading.Barrier(2)

    def work(i):
        start.wait()
        got[i] = torch.cat(feed(new_manager(1e4, **SMALL), *data[i], calls), dim=2)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    torch.cuda.synchronize()
    assert torch.equal(got[0], alone[0]) and torch.equal(got[1], alone[1])


@pytest.mark.parametrize("driven", ["resident", "host"])
@pytest.mark.parametrize("calls,kw", [([500, 1, 130], dict(SMALL)), ([500, 1], dict(SMALL, dim=32)), ([500, 1], dict(SMALL, perhead=True))],
                         ids=["128", "32", "perhead"])
def test_append_returns_contiguous_rows_on_either_path(driven, calls, kw, monkeypatch):
    """[B, H, n, D], which a caller may view with heads and tokens in one; the attention type takes the rows by token and gives
    the same ones."""
    from infllm_amd.attention import ContextManager, inf_llm_forward, RotaryEmbeddingESM
    if driven == "host":
        monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    H, Hkv, B, dim = 4, 2, 2, kw.get("dim", 128)
    q, k, v = (t.cuda() for t in make_stream(sum(calls), H, Hkv, 7, B=B, D=dim))
    outs = feed(new_manager(1e4, **kw), q, k, v, calls)
    for n, o in zip(calls, outs):
        assert o.shape == (B, H, n, dim) and o.is_contiguous() and o.view(B, H * n, dim).shape == (B, H * n, dim)
    forward = inf_llm_forward(**{n: x for n, x in kw.items() if n != "dim"}, fattn=False)
    past, pos, same = None, 0, lambda t: t
    rope = RotaryEmbeddingESM(dim, base=1e4, device="cuda")
    for n, o in zip(calls, outs):
        rows = [t[:, :, pos:pos + n].transpose(1, 2).reshape(B, n, -1) for t in (q, k, v)]
        got, past = forward(None, rows[0], rows[1], rope, True, past, same, same, lambda _: rows[2], same, dim, H, Hkv)
        assert torch.equal(got, o.transpose(1, 2).reshape(B, n, -1)) and not past.rows_by_token
        pos += n
