"""infllm_window_forward with the least scratch it takes - the rotated queries' and nothing for partial rows - against the calls of the
package, which bring more: nothing behind the scratch is written, and the results agree within their rounding to bf16 (and that of partial
rows to fp16: 2^-7 of a row's largest value)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
GUARD = 4096


class LeastScratch:
    """hands calls on with a scratch of their own, as small as it may be"""

    def __init__(self, lib, fields, block):
        self.lib, self.fields, self.block, self.rooms = lib, fields, block, []

    def infllm_window_forward(self, args, stream):
        a = dict(zip(self.fields, self.block.unpack(args)))
        size = (2 if a["kind"] else 1) * a["B"] * a["H"] * a["n_q"] * a["dim"] * 2
        room = torch.full((size + GUARD,), 0x5A, dtype=torch.uint8, device="cuda")
        a["d_work"], a["work_bytes"] = room.data_ptr(), size
        self.rooms.append((room, size))
        return self.lib.infllm_window_forward(self.block.pack(*(a[n] for n in self.fields)), stream)


@pytest.mark.parametrize("kind", ["origin", "stream-llm", "infinite-lm"])
@pytest.mark.parametrize("B,H,Hkv,D", [(1, 1, 1, 64), (1, 1, 1, 128), (1, 2, 1, 128), (2, 1, 1, 64), (1, 8, 2, 128)])
def test_the_least_scratch_is_enough(kind, B, H, Hkv, D, monkeypatch):
    from infllm_amd import _lib
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM, _sink_window
    calls, g = [150, 1, 1, 2, 3, 40, 1], torch.Generator(device="cuda").manual_seed(D + H)
    x = [torch.randn((B, sum(calls), h * D), generator=g, device="cuda").bfloat16() for h in (H, Hkv, Hkv)]
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](96, 70, fattn=False)
    rope, same = RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t

    def run():
        past, outs, at = None, [], 0
        for n in calls:
            q, k, v = (t[:, at:at + n] for t in x)
            o, past = forward(None, q, k, rope, True, past, same, same, lambda _: v, same, D, H, Hkv)
            outs.append(o.view(B, n, H, D).float())
            at += n
        return torch.cat(outs, dim=1)
    want = run()
    least = LeastScratch(_lib.load(), [n for n, _ in _lib.WindowArgs._fields_], _sink_window._ARGS)
    monkeypatch.setattr(_sink_window._lib, "load", lambda: least)
    got = run()
    for room, size in least.rooms:
        assert bool((room[size:] == 0x5A).all()), size
    assert len(least.rooms) == len(calls)
    assert bool(((got - want).abs().amax(-1) <= 2.0 ** -7 * want.abs().amax(-1)).all())
