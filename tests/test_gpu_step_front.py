"""A decode step whose prologue rides with its scores: rows of representatives of every length class these have, heads of 64
and 128, one to twelve heads a group, several batch rows, and rows too long for it - rings, books and state bit for bit those of
the host-driven path, whose prologue is a launch of its own; outputs within the difference of the key splits."""
import pytest
import torch

from stream_parity import SMALL, feed, make_stream, new_manager

pytestmark = pytest.mark.gpu

CASES = [(4, 2, 128, 1), (8, 2, 128, 2), (16, 4, 128, 1), (32, 8, 128, 1), (36, 3, 128, 2), (12, 12, 64, 1), (36, 36, 64, 1), (44, 4, 64, 1), (48, 8, 128, 1)]


@pytest.mark.parametrize("H,Hkv,D,B", CASES)
def test_steps_with_the_prologue_in_the_retrieval(H, Hkv, D, B, monkeypatch):
    from infllm_amd.attention import ContextManager
    calls, kw = [520] + [1] * 5, dict(SMALL, dim=D)
    q, k, v = (t.cuda() for t in make_stream(sum(calls), H, Hkv, 3 * H + D, B=B, D=D))
    cm = new_manager(1e4, **kw)
    got = feed(cm, q, k, v, calls)
    assert cm._resident and cm.num_global_block > kw["topk"]
    monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    ref = new_manager(1e4, **kw)
    want = feed(ref, q, k, v, calls)
    for a, b in zip(got, want):
        err = (a.float() - b.float()).abs()
        assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, float(err.max())
    assert cm.stats == ref.stats
    a, b = cm.export_state(), ref.export_state()
    for name in ("tail_k", "tail_v", "init_k", "init_v"):
        assert torch.equal(a[name], b[name]), name
    assert torch.allclose(a["tail_score"], b["tail_score"], rtol=2e-3, atol=1e-5)
