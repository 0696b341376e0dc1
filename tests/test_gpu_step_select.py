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
        ids = cm._tables.view(torch.int32)[-2 * ((B * topk + 1) // 2):][:B * topk].view(B, topk)      # the selection ends the manager's tables
        assert torch.equal(ids.long(), want), step
