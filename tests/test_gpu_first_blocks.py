"""The blocks of a stream before its first selection: a call whose blocks all lie inside the window (scored along with its merge from
1,025 up to 2,048 tokens), and blocks that attend every unit (their page tables ride in the launch of the stage, up to 64 pages over all
batch rows) - against the host-driven path: state bit for bit, outputs within the difference of the key splits, the score track
within that of their order."""
import pytest
import torch

from stream_parity import SMALL, feed, make_stream, new_manager

pytestmark = pytest.mark.gpu


def rows64(t):
    """the host-driven path's rows of 128: halves at 0 and 64"""
    return torch.cat((t[..., :32], t[..., 64:96]), dim=-1)


WINDOW = dict(SMALL, n_local=2304, exc_block_size=512)
UNITS = dict(SMALL, topk=16, max_cached_block=16)
CASES = [(n, 4, 2, 128, 1, WINDOW) for n in (1024, 1025, 2047, 2048, 2049)]
CASES += [(1025, 3, 3, 64, 2, WINDOW), (2048, 4, 1, 64, 1, WINDOW), (1900, 12, 1, 128, 2, WINDOW)]
CASES += [(700, 4, 2, 128, B, UNITS) for B in (1, 3, 4, 7)] + [(700, 2, 2, 64, 4, UNITS)]       # up to 16 or 17 pages a batch row


@pytest.mark.parametrize("n,H,Hkv,D,B,kw", CASES)
def test_blocks_before_the_first_selection(n, H, Hkv, D, B, kw, monkeypatch):
    from infllm_amd.attention import ContextManager
    calls, kw = [n, 1], dict(kw, dim=D)
    q, k, v = (t.cuda() for t in make_stream(sum(calls), H, Hkv, n + B, B=B, D=D))
    cm = new_manager(1e4, **kw)
    got = feed(cm, q, k, v, calls)
    assert cm._resident and cm.num_global_block <= kw["topk"] and (cm.num_global_block > 0) == (kw is not WINDOW and n == 700)
    monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    ref = new_manager(1e4, **kw)
    want = feed(ref, q, k, v, calls)
    assert not ref._resident
    for a, b in zip(got, want):
        err = (a.float() - b.float()).abs()
        assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, float(err.max())
    assert cm.stats == ref.stats
    T = sum(calls)                                              # (fewer than the rings hold)
    for name in ("ring_k_raw", "ring_k_rot", "ring_v"):
        assert torch.equal(getattr(cm, name)[:, :, :T, :D], getattr(ref, name)[:, :, :T, :D] if D == 128 else rows64(getattr(ref, name)[:, :, :T])), name
    assert torch.allclose(cm.ring_score[:, :, :T], ref.ring_score[:, :, :T], rtol=2e-3, atol=1e-5)
    if cm.num_global_block:
        assert torch.equal(cm.export_state()["units"], ref.export_state()["units"].cpu())
