"""Local scores where a stage of queries is masked in part: the diagonal, the far end of the window, ranges of keys that begin
and end inside a wave's, queries that end inside a stage, rings that wrap - for launches whose waves hold 32 keys and 64, of
the kernel for finished log-sum-exps and of the general one.

Against 64 bits over the same bf16 inputs and the same log-sum-exps.  A probability is exp2 of a 32-bit sum of 128 products (an
error of some 2^-20 of the logit's size, below 2^5 here) and a score a 32-bit sum of up to 600 of them: 1e-4 relative, 1e-5
absolute."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def _rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


def _visible(mask, Lq, lo, hi, offset, window):
    dist = torch.arange(Lq)[:, None] - torch.arange(lo, hi)[None, :] + offset
    return {0: torch.ones_like(dist, dtype=torch.bool), 1: (dist >= 0) & (dist < window), 2: dist >= window}[mask]


@pytest.mark.parametrize("H,Hkv,keys", [(4, 2, 700), (64, 64, 2100)])           # 32 keys a wave; 64
@pytest.mark.parametrize("Lq", [1, 33, 130, 512, 600])
@pytest.mark.parametrize("mask", ["none", "window", "complement"])
def test_scores_of_partly_masked_stages(H, Hkv, keys, Lq, mask):
    _partly_masked(H, Hkv, keys, Lq, mask)


# Two groups of waves that share a stage of 128 queries: launches of few workgroups and 256 queries or more
@pytest.mark.parametrize("Lq", [255, 256, 257, 319, 384, 385])
@pytest.mark.parametrize("mask", ["none", "window", "complement"])
def test_scores_of_paired_waves(Lq, mask):
    _partly_masked(4, 2, 900, Lq, mask)


# The general kernel, for log-sum-exps in parts: one part, fewer than eight, eight, more than a turn of eight
@pytest.mark.parametrize("H,Hkv,keys", [(4, 2, 700), (64, 64, 2100)])
@pytest.mark.parametrize("Lq,parts", [(1, 1), (33, 3), (130, 8), (512, 2), (600, 11)])
@pytest.mark.parametrize("mask", ["none", "window", "complement"])
def test_scores_of_the_general_kernel(H, Hkv, keys, Lq, parts, mask):
    _partly_masked(H, Hkv, keys, Lq, mask, parts)


def _partly_masked(H, Hkv, keys, Lq, mask, parts=0):
    from infllm_amd import _lib, ops
    cap, lo = 2304, 77
    hi = lo + keys
    code = dict(none=ops.MASK_NONE, window=ops.MASK_WINDOW, complement=ops.MASK_COMPLEMENT)[mask]
    offset, window = hi - Lq - 45, keys - 150                 # the last 45 keys behind every query, the first ones out of the window
    q, k = _rand((1, H, Lq, D), 1), _rand((1, Hkv, keys, D), 2)
    ring = torch.full((1, Hkv, cap, D), float("nan"), dtype=torch.bfloat16)
    base = 2304 * 3 - 500                                      # positions base + j, j in [lo, hi): they wrap
    rows = (torch.arange(lo, hi) + base) % cap
    ring[:, :, rows] = k
    kk = k.repeat_interleave(H // Hkv, dim=1).double()
    s = torch.matmul(q.double(), kk.transpose(2, 3).contiguous()) / math.sqrt(D) * math.log2(math.e)
    vis = _visible(code, Lq, lo, hi, offset, window)
    s = s.masked_fill(~vis, float("-inf"))
    lse = torch.logsumexp(s * math.log(2.0), -1) / math.log(2.0)
    lse32 = lse.float()
    want = torch.where(vis, torch.exp2(s - torch.where(torch.isfinite(lse), lse32.double(), math.inf)[..., None]), 0.0).sum(2)
    start = torch.rand((1, H, cap), generator=torch.Generator().manual_seed(3))
    score = start.cuda()
    where = dict(cap=cap, j_lo=base + lo, j_hi=base + hi, mask=code, offset=offset + base, window=window, accumulate=True, score_cap=cap)
    if parts:                                                  # shares of the sum; a share of nothing in the first of several
        share = torch.softmax(torch.randn((parts, 1, H, Lq), generator=torch.Generator().manual_seed(4)).double(), 0)
        if parts > 1:
            share[1] += share[0]
            share[0] = 0
        lses, q_dev, k_dev = (lse32 + torch.log2(share)).float().cuda(), q.cuda(), ring.cuda()      # (-inf where nothing is visible)
        a = ops._score_args(q_dev, k_dev, score, softmax_scale=None, **where)
        a.d_lse, a.n_parts = lses.data_ptr(), parts
        _lib.check(_lib.load().infllm_local_score(a, ops._stream()), "infllm_local_score")
    else:
        ops.local_score(q.cuda(), ring.cuda(), torch.where(torch.isfinite(lse32), lse32, math.inf).cuda(), score, **where)
    got = score.cpu()
    other = torch.ones(cap, dtype=torch.bool)
    other[rows] = False
    assert torch.equal(got[:, :, other], start[:, :, other])
    assert torch.allclose(got[:, :, rows].double(), want + start[:, :, rows].double(), rtol=1e-4, atol=1e-5), float(
        (got[:, :, rows].double() - want - start[:, :, rows].double()).abs().max())


@pytest.mark.parametrize("mask", ["window", "complement"])
@pytest.mark.parametrize("apart,window", [(2 * 10 ** 9, 15 * 10 ** 8), (2 * 10 ** 9, 2 * 10 ** 9 - 50), (6 * 10 ** 8, 6 * 10 ** 8 - 50), (2 ** 28 + 9, 2 ** 28), (2 ** 28 - 9, 2 ** 28),
                                          (2 ** 40, 2 ** 41), (-2 ** 31, 2 ** 33), (5, 2 ** 31 - 1), (-9, -5)])
def test_scores_of_keys_far_from_their_queries(apart, window, mask):
    """(positions that a caller gives: 32 bits hold neither such distances nor such windows)"""
    from infllm_amd import ops
    H, Lq, keys = 4, 70, 1100
    code = dict(window=ops.MASK_WINDOW, complement=ops.MASK_COMPLEMENT)[mask]
    q, k = _rand((1, H, Lq, D), 1), _rand((1, H, keys, D), 2)
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) / math.sqrt(D) * math.log2(math.e)
    lse = torch.logsumexp(s * math.log(2.0), -1).float() / math.log(2.0)
    want = (torch.exp2(s - lse.double()[..., None]) * _visible(code, Lq, 0, keys, apart, window)).sum(2)
    score = torch.empty((1, H, keys), device="cuda")
    ops.local_score(q.cuda(), k.cuda(), lse.cuda(), score, mask=code, offset=apart, window=window, accumulate=False)
    assert torch.allclose(score.cpu().double(), want, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("H,Hkv,keys", [(4, 2, 1025), (64, 64, 2100)])
@pytest.mark.parametrize("Lq,parts", [(1, (1, 0)), (33, (2, 1)), (512, (4, 4)), (2048, (1, 2))])
@pytest.mark.parametrize("mask", ["none", "window", "complement"])
def test_scores_with_the_merge_of_the_partials(H, Hkv, keys, Lq, parts, mask):
    """One launch against the two: rows and log-sum-exps bit for bit, scores up to the order of nothing (the same sums)."""
    from infllm_amd import ops
    if H * Lq > 64 * 512:
        H, Hkv = 4, 2
    code = dict(none=ops.MASK_NONE, window=ops.MASK_WINDOW, complement=ops.MASK_COMPLEMENT)[mask]
    where = dict(mask=code, offset=keys - Lq, window=keys - 100)
    g = torch.Generator().manual_seed(5)
    q, k = _rand((2, H, Lq, D), 1).cuda(), _rand((2, Hkv, keys, D), 2).cuda()
    sets = [p for p in parts if p]
    o_parts = [torch.randn((p, 2, H, Lq, D), generator=g).half().cuda() for p in sets]
    lse_parts = [(4 + torch.randn((p, 2, H, Lq), generator=g)).cuda() for p in sets]
    out, lse, score = (torch.empty((2, H, Lq, D), dtype=torch.bfloat16, device="cuda"), torch.empty((2, H, Lq), device="cuda"),
                       torch.empty((2, H, keys), device="cuda"))
    assert ops.merge_sets_and_score(o_parts, lse_parts, out, lse, q, k, score, **where)
    want_out, want_lse, want = torch.empty_like(out), torch.empty_like(lse), torch.empty_like(score)
    ops.attn_merge_sets(o_parts, lse_parts, want_out, want_lse)
    ops.local_score(q, k, want_lse, want, accumulate=False, **where)
    assert torch.equal(out, want_out) and torch.equal(lse, want_lse)
    assert torch.allclose(score, want, rtol=1e-6, atol=0)
    for lse_part, o_part in zip(lse_parts, o_parts):             # a query whose logits are no numbers: empty sums, rows of NaN
        lse_part[:, :, :, Lq // 2], o_part[:, :, :, Lq // 2] = -math.inf, math.nan
    assert ops.merge_sets_and_score(o_parts, lse_parts, out, lse, q, k, score, **where)
    ops.attn_merge_sets(o_parts, lse_parts, want_out, want_lse)
    ops.local_score(q, k, want_lse, want, accumulate=False, **where)
    assert out[:, :, Lq // 2].isnan().all() and torch.allclose(out.float(), want_out.float(), rtol=0, atol=0, equal_nan=True) and torch.equal(lse, want_lse)
    assert torch.allclose(score, want, rtol=1e-6, atol=0, equal_nan=True) and (mask == "complement" or not score.isfinite().all())
    small = torch.empty((2, H, 1024), device="cuda")
    assert not ops.merge_sets_and_score(o_parts, lse_parts, out, lse, q, k[:, :, :1024], small, **where)       # (too few keys)
