"""Steps of the sliding-window and causal types in HIP graphs: two graphs captured on one stream whose eager steps have run before,
replayed on two streams at once, beside eager steps, several times.  Every replay's output is bit for bit that of the two launches
that a captured step takes; eager steps are within the rounding of fp16 partial rows at other split boundaries and of the result to
bf16 (2^-7 of a row's largest value)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
H, HKV, D = 16, 4, 128


@pytest.mark.parametrize("kind,past", [("origin", 700), ("stream-llm", 90), ("stream-llm", 700), ("infinite-lm", 700)])
def test_replays_beside_each_other_and_beside_eager_steps(kind, past, monkeypatch):
    from infllm_amd.attention import ATTN_FORWRAD, RotaryEmbeddingESM, _sink_window
    g = torch.Generator(device="cuda").manual_seed(past)
    x = [torch.randn((1, past + 1, h * D), generator=g, device="cuda").bfloat16() for h in (H, HKV, HKV)]
    forward = ATTN_FORWRAD[kind](False) if kind == "origin" else ATTN_FORWRAD[kind](96, 16, fattn=False)
    rope, same = RotaryEmbeddingESM(D, base=1e4, device="cuda"), lambda t: t

    def call(lo, hi, cache):
        q, k, v = (t[:, lo:hi] for t in x)
        return forward(None, q, k, rope, True, cache, same, same, lambda _: v, same, D, H, HKV)
    _, prompt = call(0, past, None)
    with monkeypatch.context() as m:
        m.setattr(_sink_window, "_ticket", lambda *_: 0)
        want, _ = call(past, past + 1, prompt)
    capture, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(capture):
        eager, _ = call(past, past + 1, prompt)                        # the stream's words are there
    torch.cuda.synchronize()
    graphs, outs = [], []
    for _ in range(2):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=capture):
            outs.append(call(past, past + 1, prompt)[0])
    for _ in range(3):
        for out in outs:
            out.zero_()
        torch.cuda.synchronize()
        for stream, graph in zip((capture, other), graphs):
            with torch.cuda.stream(stream):
                graph.replay()
        with torch.cuda.stream(capture):
            eager, _ = call(past, past + 1, prompt)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], want) and torch.equal(outs[1], want)
        a, b = (t.view(H, D).float() for t in (eager, want))
        assert bool(((a - b).abs().amax(-1) <= 2.0 ** -7 * b.abs().amax(-1)).all())
