"""The launch that ends a block (scores, merge, the units that leave, the next block's ranking) in the forms it takes: units of
every size it has, units of two chunks, blocks behind which nothing leaves, short last blocks, several batch rows, heads of 64,
rows of representatives that are ranked by a launch of their own - against the host-driven path, whose launches do one thing each."""
import pytest
import torch

from stream_parity import REFERENCE, feed, make_stream, new_manager

pytestmark = pytest.mark.gpu
KW = dict(REFERENCE, n_local=1100, n_init=64, topk=6, max_cached_block=16, repr_topk=3)

CASES = [
    ("units of 32", [2600, 700], 8, 2, 1, dict(KW, block_size=32)),
    ("units of 64", [2600, 700], 8, 2, 2, dict(KW, block_size=64)),
    ("units of 96", [3300, 513], 8, 2, 1, dict(KW, block_size=96)),
    ("units of 128, one head", [3500, 600], 1, 1, 2, dict(KW, block_size=128)),
    ("units of 48: launches of their own", [2600, 300], 8, 2, 1, dict(KW, block_size=48)),
    ("blocks that carve nothing", [2600, 200], 8, 2, 1, dict(KW, block_size=128, exc_block_size=64)),
    ("short blocks, no sinks", [2400, 333], 4, 4, 1, dict(KW, block_size=64, exc_block_size=96, n_init=0)),
    ("long rows", [3300, 300], 40, 8, 1, dict(KW, block_size=128)),
    ("heads of 64", [2900, 700], 6, 3, 2, dict(KW, block_size=64, dim=64)),
    ("44 heads of 64", [2900, 300], 44, 44, 1, dict(KW, block_size=128, dim=64)),
]


@pytest.mark.parametrize("name,calls,H,Hkv,B,kw", CASES, ids=[c[0] for c in CASES])
def test_blocks_end_as_they_do_launch_by_launch(name, calls, H, Hkv, B, kw, monkeypatch):
    import infllm_amd.attention.context_manager as manager_module
    from infllm_amd.attention import ContextManager
    monkeypatch.setattr(manager_module, "_UNIT_CHUNK", 6)           # (blocks of four units end in the middle of one)
    T = sum(calls)
    q, k, v = (t.cuda() for t in make_stream(T, H, Hkv, 9 + T, B=B, D=kw.get("dim", 128)))
    cm = new_manager(1e4, **kw)
    got = feed(cm, q, k, v, calls)
    assert cm._resident and cm.num_global_block > kw["topk"] and cm.stats["misses"] > 0
    assert int(cm._call_buf["ticket"].item()) == 0
    monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    ref = new_manager(1e4, **kw)
    want = feed(ref, q, k, v, calls)
    assert not ref._resident
    for n, a, b in zip(calls, got, want):
        if kw.get("dim") != 64 and kw["exc_block_size"] != 96:      # the same kernels and splits: the same bits
            assert torch.equal(a, b), n
        err = (a.float() - b.float()).abs()
        assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, (n, float(err.max()))
    assert cm.stats == ref.stats
    a, b = cm.export_state(), ref.export_state()
    assert torch.equal(a["units"], b["units"].cpu()) and torch.equal(a["reps"].cpu(), b["reps"].cpu())
    assert torch.allclose(a["tail_score"], b["tail_score"], rtol=2e-3, atol=1e-5)


@pytest.mark.parametrize("H,Hkv,D,B", [(8, 2, 128, 1), (6, 3, 64, 2), (40, 8, 128, 1)])
def test_blocks_behind_more_chunks_of_units_than_a_ranking_keeps_addresses_of(H, Hkv, D, B, monkeypatch):
    """A chunk for every unit, and more units than the 256 whose addresses a ranking workgroup reads ahead (rows of 40 x 128: a launch of
    its own ranks): the same bits as with a few large chunks."""
    import infllm_amd.attention.context_manager as manager_module
    calls, kw = [5120, 5120, 1, 1100], dict(KW, block_size=32, dim=D, exc_block_size=256)
    q, k, v = (t.cuda() for t in make_stream(sum(calls), H, Hkv, 11, B=B, D=D))

    def run(unit_chunk):
        monkeypatch.setattr(manager_module, "_UNIT_CHUNK", unit_chunk)
        cm = new_manager(1e4, **kw)
        return cm, feed(cm, q, k, v, calls)
    cm, got = run(1)
    ref, want = run(64)
    assert cm._resident and ref._resident and len(cm._chunks) == cm.num_global_block > 300 and len(ref._chunks) < 10
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert cm.stats == ref.stats and all(a.cached == b.cached for a, b in zip(cm.policy, ref.policy))
    assert torch.equal(cm.export_state()["units"], ref.export_state()["units"])
