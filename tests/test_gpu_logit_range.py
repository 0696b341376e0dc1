"""Logits far from zero: the running max moves by hundreds of powers of two - rows whose keys' logits all lie
high or low, keys whose logits rise or fall by more than the range of an exponent behind each other, one key above or below all others.

Against a dense softmax in 64 bits over the same bf16 inputs, or the oracle's in 32 bits, max-abs 2e-2 / mean-abs 2e-3 as in the other
tests: products of up to 300 are summed in 32 bits by 8 MFMAs in a row (of 16 elements), whose sums round by
300 x 2^-24 each: 1.4e-4 of a probability at worst."""
import pytest
import torch

from oracle.rope import RopeOracle
from oracle.siblings import CausalOracle, SinkWindowOracle
from test_gpu_attn_tiles import _check, _dense, _partials, _rand

pytestmark = pytest.mark.gpu

# what is added to the logit of key j of n (in nats, exact in bf16)
SHIFTS = {
    "high": lambda j, n: 100.0,
    "low": lambda j, n: -120.0,
    "rising": lambda j, n: 200.0 if j >= n // 2 else -40.0,
    "falling": lambda j, n: -200.0 if j >= n // 2 else 40.0,
    "one key": lambda j, n: 128.0 if j == n // 3 else 0.0,
    "low but one": lambda j, n: 0.0 if j == n // 3 else -100.0,
}


def _shifted(q, k, shift, heads, dim, last):
    """Adds shift(j) to the logits of the given heads: one component, the same in every query, carries it."""
    n = k.shape[2]
    q[..., last], k[..., last] = 0.0, torch.tensor([shift(j, n) for j in range(n)]).bfloat16()
    q[:, heads, :, last] = 8.0 if dim == 64 else 11.3125                       # (about sqrt(dim))
    return q, k


@pytest.mark.parametrize("what", SHIFTS)
@pytest.mark.parametrize("heads", [slice(None), slice(1, 2)], ids=["all heads", "one head"])
def test_stages(what, heads):
    from infllm_amd import ops
    B, H, Hkv, Lq, n = 1, 8, 2, 70, 576
    q, k, v = _rand((B, H, Lq, 128), 7), _rand((B, Hkv, n, 128), 8), _rand((B, Hkv, n, 128), 9)
    _shifted(q, k, SHIFTS[what], heads, 128, 127)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    pages = ops.make_pages([(kd[0, 0, 64 * p:].data_ptr(), vd[0, 0, 64 * p:].data_ptr(), n * 128, 64) for p in range(n // 64)])
    pages = torch.frombuffer(bytearray(pages), dtype=torch.uint8).cuda()
    for ns in (1, 2):
        for window in (0, 200, 1 << 40):
            o_part, lse_part = _partials(ns, B, H, Lq)
            ops.attn_stage_linear(qd, kd, vd, o_part, lse_part, cap=n, j_lo=0, j_hi=n, mask=int(window > 0), offset=n - Lq, window=window, nsplit=ns)
            out, lse = torch.empty((B, H, Lq, 128), dtype=torch.bfloat16, device="cuda"), torch.empty((B, H, Lq), device="cuda")
            ops.attn_merge(o_part, lse_part, ns, out, lse)
            dist = torch.arange(Lq)[:, None] + n - Lq - torch.arange(n)[None, :]
            vis = (dist >= 0) & (dist < window) if window else torch.ones_like(dist, dtype=torch.bool)
            _check(out, lse, *_dense(q, k, v, vis), (ns, window))
        o_part, lse_part = _partials(ns, B, H, Lq)
        ops.attn_stage_paged(qd, pages, n // 64, Hkv, o_part, lse_part, nsplit=ns)
        ops.attn_merge(o_part, lse_part, ns, out, lse)
        _check(out, lse, *_dense(q, k, v, torch.ones((Lq, n), dtype=torch.bool)), (ns, "pages"))


@pytest.mark.parametrize("what", SHIFTS)
@pytest.mark.parametrize("kind", ["origin", "infinite-lm", "stream-llm"])
@pytest.mark.parametrize("dim,H,Hkv", [(128, 8, 2), (64, 8, 2), (64, 3, 3)])
def test_window_types(what, kind, dim, H, Hkv):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM
    n, n_local, n_init, base = 777, 300, 8, 1e30                        # (of that base the last pair does not turn)
    g = torch.Generator().manual_seed(dim)
    q, k, v = (torch.randn(1, h, n, dim, generator=g).bfloat16() for h in (H, Hkv, Hkv))
    q[..., dim // 2 - 1] = k[..., dim // 2 - 1] = 0.0
    _shifted(q, k, SHIFTS[what], slice(None), dim, dim - 1)
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](n_local, n_init, fattn=False)
    rope = RopeOracle(dim, base=base)
    ora = CausalOracle(rope) if kind == "origin" else SinkWindowOracle(rope, n_local, n_init, kind)
    past, same = None, lambda t: t
    rows = lambda t, a, b: t[:, :, a:b].transpose(1, 2).reshape(1, b - a, -1).cuda()
    for a, b in ((0, 400), (400, n)):
        got, past = forward(None, rows(q, a, b), rows(k, a, b), RotaryEmbeddingESM(dim, base=base, device="cuda"), True, past, same, same,
                            lambda _: rows(v, a, b), same, dim, H, Hkv)
        err = (got.view(1, b - a, H, dim).transpose(1, 2).float().cpu() - ora.append(q[:, :, a:b].float(), k[:, :, a:b].float(), v[:, :, a:b].float())).abs()
        assert float(err.max()) <= 2e-2 and float(err.mean()) <= 2e-3, (a, float(err.max()), float(err.mean()))
