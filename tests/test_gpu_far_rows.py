"""Keys and values whose rows lie far apart - every n-th row of a long tensor, layouts with the heads inside the rows -, at distances
where a tile of 64 rows spans more than 2^32 bytes: bit for bit what the same rows give next to each other.  And queries whose rows
are given backwards (a negative stride), which an offset of 32 bits without a sign does not reach."""
import pytest
import torch

pytestmark = pytest.mark.gpu
H, HKV, D = 4, 2, 128


def _far(rows, sl, seed):
    """[1, HKV, rows, D] with its rows sl elements apart, and the same next to each other"""
    near = torch.randn((1, HKV, rows, D), generator=torch.Generator().manual_seed(seed)).bfloat16().cuda()
    room = torch.empty(((rows - 1) * sl + HKV * D,), dtype=torch.bfloat16, device="cuda")
    far = room.as_strided((1, HKV, rows, D), (room.numel() // 8 * 8, D, sl, 1))
    far.copy_(near)
    return far, near


@pytest.mark.parametrize("rows,k_sl,v_sl", [(130, 2 ** 25, 256), (130, 2 ** 25 - 8, 2 ** 25 + 8), (75, 2 ** 26, 2 ** 26), (64, 2 ** 26 + 8, 256), (13, 2 ** 27 - 8, 2 ** 27 - 8), (13, 256, 2 ** 27),
                                            (2, 2 ** 31 + 8, 2 ** 30), (1, 2 ** 35, 2 ** 33)])
@pytest.mark.parametrize("window", [None, 40])
def test_rows_far_apart(rows, k_sl, v_sl, window):
    from infllm_amd.attention.dot_production_attention import get_multi_stage_dot_production_attention
    operator, _ = get_multi_stage_dot_production_attention(False)
    q = torch.randn((1, H, 37, D), generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    (k, near_k), (v, near_v) = _far(rows, k_sl, 2), _far(rows, v_sl, 3)

    def result(k, v):
        a = operator(q.shape, q.dtype, q.device)
        a.append(q, k, v, sliding_window=window, get_score=True, end=True)
        return a.get_result()
    (out, (score,)), (want, (want_score,)) = result(k, v), result(near_k, near_v)
    assert torch.equal(out, want) and torch.equal(score, want_score)


@pytest.mark.parametrize("Lq", [2, 33, 100])
@pytest.mark.parametrize("H,keys", [(4, 300), (64, 2100)])
def test_queries_given_backwards(H, keys, Lq):
    from infllm_amd import _lib, ops
    q, k, v = (torch.randn((1, h, n, D), generator=torch.Generator().manual_seed(i)).bfloat16().cuda() for i, (h, n) in enumerate(((H, Lq), (HKV, keys), (HKV, keys))))
    back = q.flip(2).contiguous()
    parts = lambda: (torch.empty((1, 1, H, Lq, D), dtype=torch.float16, device="cuda"), torch.empty((1, 1, H, Lq), device="cuda"))
    (o, lse), (want_o, want_lse) = parts(), parts()
    ops.attn_stage_linear(q, k, v, want_o, want_lse)
    a = ops.linear_stage_args(back, k, v, o, lse)
    a.d_q, a.q_sl = back.data_ptr() + (Lq - 1) * D * 2, -D
    _lib.check(_lib.load().infllm_attn_stage(a, ops._stream()), "infllm_attn_stage")
    assert torch.equal(o, want_o) and torch.equal(lse, want_lse)
    scores = [torch.empty((1, H, keys), device="cuda") for _ in range(2)]
    ops.local_score(q, k, want_lse[0], scores[0], accumulate=False)
    s = ops._score_args(back, k, scores[1], None, 0, None, ops.MASK_NONE, 0, 0, False, None, None)
    s.d_q, s.q_sl, s.d_lse = back.data_ptr() + (Lq - 1) * D * 2, -D, want_lse.data_ptr()
    _lib.check(_lib.load().infllm_local_score(s, ops._stream()), "infllm_local_score")
    assert torch.allclose(scores[1], scores[0], rtol=1e-5, atol=0)          # (another kernel: 32-bit sums of up to 100 terms in another order)
