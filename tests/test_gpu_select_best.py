"""The selection behind a retrieval's last score, at the edges of its forms: 4, 16 or 32 units a thread of 512, up to 16 units or more, few
units for as many, equal scores, infinities.  Rows of one component times a query of ones there: scores are exact, and so are the ids of a
stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu

VALUES = {
    "normal": lambda n, g: torch.randn(n, generator=g),
    "equal": lambda n, g: torch.full((n,), 2.5),
    "two values": lambda n, g: torch.randint(0, 2, (n,), generator=g).float(),
    "one above": lambda n, g: torch.cat([torch.full((n - 1,), -3.0), torch.tensor([5.0])]),
    "far apart": lambda n, g: torch.randn(n, generator=g) * 10.0 ** torch.randint(-30, 30, (n,), generator=g),
    "infinite": lambda n, g: torch.where(torch.rand(n, generator=g) < 0.2, torch.tensor(float("inf")), torch.randn(n, generator=g)),
}


@pytest.mark.parametrize("what", VALUES)
@pytest.mark.parametrize("units", [17, 64, 65, 128, 129, 512, 513, 2047, 2048, 2049, 8192, 8193, 16384])
def test_the_best_units_in_order(units, what):
    from infllm_amd import ops
    g = torch.Generator().manual_seed(units)
    value = VALUES[what](units, g).bfloat16()
    reps = torch.zeros((units, 512), dtype=torch.bfloat16)
    reps[:, 0] = value
    query = torch.zeros(512)
    query[0] = 1.0
    reps, query = reps.cuda(), query.cuda()
    order = torch.sort(value.float(), descending=True, stable=True).indices
    for k in (1, 8, 16, 17, 32, 33, 64):
        if k > units:
            continue
        scores, idx = torch.empty(units, device="cuda"), torch.empty(k, dtype=torch.int32, device="cuda")
        ops.score_topk(reps, units, query, k, scores, idx)
        assert torch.equal(scores.cpu(), value.float()), k
        assert idx.cpu().tolist() == order[:k].tolist(), k
