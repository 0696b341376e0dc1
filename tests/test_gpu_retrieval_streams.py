"""Retrievals that run beside each other: on two streams far ahead of the GPU, and in graphs that are replayed on another stream than
the one they were captured on.  Scores and ids bit for bit those of a retrieval by itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu
C, K = 1024, 16


def _case(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((n, C), generator=g, device="cuda").bfloat16(), torch.randn((C,), generator=g, device="cuda"), n


def _room(n, runs=1):
    return torch.full((runs, n), -1.0, device="cuda"), torch.full((runs, K), -1, dtype=torch.int32, device="cuda")


def _alone(case):
    from infllm_amd import ops
    reps, query, n = case
    scores, idx = _room(n)
    ops.unit_scores(reps, 0, n, query, scores[0])
    ops.topk(scores[0], n, K, idx[0])
    torch.cuda.synchronize()
    return scores[0], idx[0]


def _same(room, want):
    return all(torch.equal(got, w.expand_as(got)) for got, w in zip(room, want))


@pytest.mark.parametrize("sizes", [(3000, 5000), (16384, 64)])
def test_streams_and_graphs_beside_each_other(sizes):
    from infllm_amd import ops
    cases = [_case(n, n) for n in sizes]
    wants = [_alone(case) for case in cases]
    streams = [torch.cuda.Stream() for _ in cases]
    graphs, captured = [], []
    for (reps, query, n), stream in zip(cases, streams):
        with torch.cuda.stream(stream):
            ops.score_topk(reps, n, query, K, *(t[0] for t in _room(n)))                # (a warm-up on the stream of the capture)
        torch.cuda.synchronize()
        captured.append(_room(n))
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=stream):
            ops.score_topk(reps, n, query, K, *(t[0] for t in captured[-1]))
    for _ in range(3):
        eager = [_room(n, 100) for _, _, n in cases]
        for room in captured:
            room[0].fill_(-1), room[1].fill_(-1)
        torch.cuda.synchronize()
        for i in range(100):
            for j, (reps, query, n) in enumerate(cases):
                with torch.cuda.stream(streams[j]):
                    if i % 10 == 5:
                        graphs[1 - j].replay()
                    ops.score_topk(reps, n, query, K, *(t[i] for t in eager[j]))
        torch.cuda.synchronize()
        for room, kept, want in zip(eager, captured, wants):
            assert _same(room, want) and _same(kept, want)

