"""A decode step whose attention selects the units itself: the ids it leaves are the best of the step's scores, best first and equal
scores by ascending id, at the sizes where the selection's rounds, groups and survivors change."""
import pytest
import torch

from stream_parity import new_manager

pytestmark = pytest.mark.gpu

# units, units selected, batch, representatives: of all values, all the same (every unit passes the threshold, more than are kept),
# falling with the unit's number, a few values
CASES = [(2, 1, 1, "any"), (17, 16, 1, "any"), (18, 17, 2, "any"), (65, 64, 1, "any"), (255, 16, 1, "any"), (256, 32, 1, "any"), (257, 33, 2, "any"),
         (2048, 16, 1, "any"), (2049, 64, 1, "any"), (9000, 16, 1, "any"), (16384, 64, 1, "any"), (16384, 16, 1, "falling"), (512, 16, 1, "same"),
         (513, 16, 2, "same"), (3000, 64, 1, "same"), (700, 5, 1, "few")]


@pytest.mark.parametrize("units,topk,B,how", CASES)
def test_a_step_selects_the_best_units(units, topk, B, how):
    H, Hkv, D, bs, n_init, n_local = 4, 2, 128, 8, 8, 64
    g = torch.Generator(device="cuda").manual_seed(units + topk)
    bf = lambda *s: torch.randn(s, generator=g, device="cuda").bfloat16()
    reps = bf(B, units, H * D)
    if how == "same":
        reps[:] = reps[:, :1]
    elif how == "falling":                                    # multiples of the first row
        reps = reps[:, :1] * torch.linspace(1, -1, units, device="cuda")[None, :, None].bfloat16()
    elif how == "few":
        reps = reps[:, torch.randint(0, 4, (units,), generator=g, device="cuda")]
    cm = new_manager(1e4, n_init=n_init, n_local=n_local, block_size=bs, max_cached_block=64, topk=topk, exc_block_size=32, repr_topk=1)
    cm.load_state(dict(length=n_init + units * bs + n_local, tail_k=bf(B, Hkv, n_local, D), tail_v=bf(B, Hkv, n_local, D), tail_score=None,
                       init_k=bf(B, Hkv, n_init, D), init_v=bf(B, Hkv, n_init, D), units=bf(units, B, 2, Hkv, bs, D), reps=reps))
    for step in range(3):
        q, k, v = bf(B, H, 1, D), bf(B, Hkv, 1, D), bf(B, Hkv, 1, D)
        assert torch.isfinite(cm.append(q, k, v, q, k, v)).all()
        scores = cm.unit_scores[:, :units]
        want = torch.sort(scores, dim=1, descending=True, stable=True).indices[:, :topk]
        torch.cuda.synchronize()
        log = cm._log.view(-1, B * topk + 1)                  # (infllm_resident_desc: log_slots x (the selection, its sequence number))
        ids = log[log[:, -1].argmax(), :-1].view(B, topk)
        assert torch.equal(ids.long(), want.cpu()), step


@pytest.mark.parametrize("units,H,Hkv,D,B", [(2500, 4, 1, 128, 34), (2100, 36, 36, 64, 1), (4500, 8, 8, 64, 5), (2049, 33, 33, 128, 1), (2300, 32, 32, 128, 1)])
def test_prologues_of_many_heads_beside_the_scores(units, H, Hkv, D, B, monkeypatch):
    """More (batch row, kv head) pairs than the scores leave places for (32 of 256), behind units that fill them; and 32, which they do:
    scores of every batch row, the books, the rows and the score track, against the host-driven path."""
    from infllm_amd.attention import ContextManager
    bs, n_init, n_local, topk = 8, 8, 64, 16
    g = torch.Generator(device="cuda").manual_seed(units + B)
    bf = lambda *s: torch.randn(s, generator=g, device="cuda").bfloat16()
    state = dict(length=n_init + units * bs + n_local, tail_k=bf(B, Hkv, n_local, D), tail_v=bf(B, Hkv, n_local, D), tail_score=None, init_k=bf(B, Hkv, n_init, D),
                 init_v=bf(B, Hkv, n_init, D), units=bf(units, B, 2, Hkv, bs, D), reps=bf(B, units, H * D))
    steps = [(bf(B, H, 1, D), bf(B, Hkv, 1, D), bf(B, Hkv, 1, D)) for _ in range(3)]

    def manager():
        cm = new_manager(1e4, n_init=n_init, n_local=n_local, block_size=bs, max_cached_block=64, topk=topk, exc_block_size=32, repr_topk=1, dim=D)
        return cm.load_state(state), [cm.append(*step, *step) for step in steps]
    cm, got = manager()
    monkeypatch.setattr(ContextManager, "resident_bytes", 0)
    ref, want = manager()
    assert cm._resident and not ref._resident
    for a, b in zip(got, want):
        err = (a.float() - b.float()).abs()
        assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, float(err.max())
    # 32-bit sums of H * D products of N(0, 1) and a rotated N(0, 1), in another order: partial sums of the order of (H * D) ** 0.5, in
    # chains of some 64
    assert float((cm.unit_scores[:, :units] - ref.unit_scores[:, :units]).abs().max()) <= (H * D) ** 0.5 * 64 * 2.0 ** -23
    assert cm.stats == ref.stats and all(a.cached == b.cached for a, b in zip(cm.policy, ref.policy))
    a, b = cm.export_state(), ref.export_state()
    for name in ("tail_k", "tail_v", "init_k", "init_v"):
        assert torch.equal(a[name], b[name]), name
    assert torch.allclose(a["tail_score"], b["tail_score"], rtol=2e-3, atol=1e-5)
