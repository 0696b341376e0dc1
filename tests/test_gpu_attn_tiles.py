"""The tile loop of the attention kernel at the ends of its lists: a tile is worked off in two turns, the one after next is
requested meanwhile, and tiles with nothing special about them take a form of their own - so lists of one to nine tiles,
splits in the middle of them, rings that wrap at any tile, ranges that begin and end inside tiles and pages with missing rows.

Against a dense softmax in 64 bits over the same bf16 inputs, max-abs 2e-2 / mean-abs 2e-3 (the probabilities are rounded
to bf16: a relative 2^-9 of values up to 4 or 5)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def _rand(shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).bfloat16()


def _dense(q, k, v, visible):
    """[B,H,Lq,D] against [B,Hkv,L,D] under visible [Lq, L]; rows that see nothing are 0 with log-sum-exp -inf (base 2)."""
    G = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(G, dim=1) for t in (k, v))
    s = torch.matmul(q.double(), k.transpose(2, 3).contiguous()) / math.sqrt(D) * math.log2(math.e)
    s = s.masked_fill(~visible, float("-inf"))
    m = s.amax(-1, keepdim=True).clamp_min(-1e300)
    p = torch.exp2(s - m)
    den = p.sum(-1, keepdim=True)
    out = torch.where(den > 0, torch.matmul(p, v) / den.clamp_min(1e-300), torch.zeros((), dtype=torch.float64))
    return out, (m + torch.log2(den)).squeeze(-1)


def _check(out, lse, want, want_lse, what):
    err = (out.double().cpu() - want).abs()
    assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, (what, float(err.max()), float(err.mean()))
    seen = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse.cpu()), seen), what
    if bool(seen.any()):
        assert float((lse.cpu().double() - want_lse)[seen].abs().max()) <= 2e-2, what


def _partials(ns, B, H, Lq):
    return (torch.empty((ns, B, H, Lq, D), dtype=torch.float16, device="cuda"), torch.empty((ns, B, H, Lq), device="cuda"))


@pytest.mark.parametrize("H,Hkv,Lq", [(8, 2, 70), (4, 4, 33), (1, 1, 300)])
@pytest.mark.parametrize("nsplit", [1, 2, 3])
def test_linear_lists_of_one_to_nine_tiles(H, Hkv, Lq, nsplit):
    from infllm_amd import ops
    B, cap, T = 2, 640, 2000
    q, k, v = _rand((B, H, Lq, D), 1), _rand((B, Hkv, T, D), 2), _rand((B, Hkv, T, D), 3)
    ring_k, ring_v = (torch.full((B, Hkv, cap, D), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    for n, (lo, hi) in enumerate([(130, 194), (128, 192), (577, 650), (640, 830), (100, 290), (700, 960), (513, 833), (1020, 1404), (1279, 1727), (1001, 1577)]):
        rows = torch.arange(lo, hi)
        ring_k.fill_(float("nan")), ring_v.fill_(float("nan"))          # rows outside the range must not be multiplied with
        ring_k[:, :, rows % cap], ring_v[:, :, rows % cap] = k[:, :, rows], v[:, :, rows]
        for mask, offset, window in ((0, 0, 0), (1, hi - Lq, 1 << 40), (1, hi - Lq, 150), (1, (lo + hi) // 2, 64), (2, hi, 100)):
            dist = torch.arange(Lq)[:, None] + offset - rows[None, :]
            vis = torch.ones_like(dist, dtype=torch.bool) if mask == 0 else (dist >= 0) & (dist < window) if mask == 1 else dist >= window
            o_part, lse_part = _partials(nsplit, B, H, Lq)
            ops.attn_stage_linear(q.cuda(), ring_k.cuda(), ring_v.cuda(), o_part, lse_part, cap=cap, j_lo=lo, j_hi=hi, mask=mask, offset=offset,
                                  window=window, nsplit=nsplit)
            out, lse = torch.empty((B, H, Lq, D), dtype=torch.bfloat16, device="cuda"), torch.empty((B, H, Lq), device="cuda")
            ops.attn_merge(o_part, lse_part, nsplit, out, lse)
            _check(out, lse, *_dense(q, k[:, :, rows], v[:, :, rows], vis), (lo, hi, mask, offset, window))


@pytest.mark.parametrize("valid", [[64], [3], [64, 64], [64, 64, 64, 64, 64, 64, 64], [64, 1, 64, 64, 64, 64], [64] * 5 + [40], [20, 64, 64, 64, 33, 64, 64, 64, 7],
                                   [64] * 9])
@pytest.mark.parametrize("nsplit", [1, 2, 3])
def test_page_lists_of_one_to_nine_tiles(valid, nsplit):
    from infllm_amd import ops
    B, H, Hkv, Lq, n = 2, 8, 2, 70, len(valid)
    q, k, v = _rand((B, H, Lq, D), 4), _rand((B, n, Hkv, 64, D), 5), _rand((B, n, Hkv, 64, D), 6)
    for p, rows in enumerate(valid):
        k[:, p, :, rows:], v[:, p, :, rows:] = float("nan"), float("nan")
    kd, vd = k.cuda(), v.cuda()
    arr = ops.make_pages([(kd[b, p].data_ptr(), vd[b, p].data_ptr(), 64 * D, valid[p]) for b in range(B) for p in range(n)])
    pages = torch.frombuffer(bytearray(arr), dtype=torch.uint8).cuda()
    o_part, lse_part = _partials(nsplit, B, H, Lq)
    ops.attn_stage_paged(q.cuda(), pages, n, Hkv, o_part, lse_part, nsplit=nsplit)
    out, lse = torch.empty((B, H, Lq, D), dtype=torch.bfloat16, device="cuda"), torch.empty((B, H, Lq), device="cuda")
    ops.attn_merge(o_part, lse_part, nsplit, out, lse)
    flat = lambda t: torch.cat([t[:, p, :, :r] for p, r in enumerate(valid)], dim=2)
    _check(out, lse, *_dense(q, flat(k), flat(v), torch.ones((Lq, sum(valid)), dtype=torch.bool)), valid)
