"""One prepared decode launch on several streams and in several captured graphs
at once: every stream and every capture has a workspace and merge counters of
its own, for partitions, balanced runs and launches without either.

Tolerances: bit for bit against the same plan run alone (the partitions and
their merge order are fixed), and ``tests/_parity.py`` against the fp32 oracle.
"""

from __future__ import annotations

import pytest
import torch

from _parity import assert_parity, make_paged, make_query
from flashattntile_amd import DecodeLaunch, PagedKVCache, _hip
from flashattntile_amd.kernels import decode as dec
from oracle.reference import ref_attention_paged

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [3000, 2100, 17, 900, 1, 2999, 64, 640]
CONFIGS = [{"split_k": 4}, {"split_k": 20}, {"balanced": 1}, {"split_k": 1}]


def _setup(P=16, queries=4):
    k, v, pt, sl = make_paged(LENS, 8, 128, P, torch.float16, seed=7, device=DEV)
    cache = PagedKVCache(k, v, pt, sl, P)
    qs = [make_query(len(LENS), 32, 128, torch.float16, seed=20 + i, device=DEV) for i in range(queries)]
    refs = [ref_attention_paged(q.cpu().float(), k.cpu().float(), v.cpu().float(), pt.cpu(), sl.cpu(),
                                return_fp32=True) for q in qs]
    return cache, qs, refs


@pytest.mark.parametrize("config", CONFIGS)
def test_plan_on_several_streams(config):
    print(f"plan on several streams {config}", flush=True)
    cache, qs, refs = _setup()
    plan = DecodeLaunch(qs[0], cache, config=config)
    alone = [plan.run(q).clone() for q in qs]
    streams = [torch.cuda.Stream() for _ in qs]
    outs = [[torch.empty_like(q) for _ in range(20)] for q in qs]
    torch.cuda.synchronize()
    for i in range(20):
        for n, s in enumerate(streams):
            with torch.cuda.stream(s):  # torch's current stream, and a handle
                plan.run(qs[n], outs[n][i]) if i % 2 else plan.run(qs[n], outs[n][i], stream=s.cuda_stream)
    torch.cuda.synchronize()
    for n, ref in enumerate(refs):
        assert_parity(alone[n], ref, label=f"streams {config}")
        for i, out in enumerate(outs[n]):
            assert torch.equal(out, alone[n]), (n, i)
    states = [plan._state(s.cuda_stream) for s in streams] + [plan._state(_hip.current_stream_handle(qs[0].device))]
    assert states[-1].workspace is plan.workspace and states[-1].counters is plan.counters
    assert (plan.workspace is None) == (config == {"split_k": 1})
    if plan.workspace is not None:
        spans = sorted((t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for s in states
                       for t in (s.workspace, s.counters))
        assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
        assert all(int(s.counters.abs().max()) == 0 for s in states)


@pytest.mark.parametrize("config", CONFIGS)
def test_graphs_of_one_plan_replay_together(config):
    """Six graphs (more than have cleared counters ready) captured from one
    plan, replayed on streams of their own beside eager runs; a stream that
    captured runs eagerly afterwards."""
    print(f"graphs of one plan {config}", flush=True)
    cache, qs, refs = _setup(queries=7)
    plan = DecodeLaunch(qs[0], cache, config=config)
    alone = [plan.run(q).clone() for q in qs]
    side = torch.cuda.Stream()
    graphs, outs = [], [torch.empty_like(q) for q in qs]
    for n in range(6):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            plan.run(qs[n], outs[n])
        graphs.append((graph, torch.cuda.Stream()))
    with torch.cuda.stream(side):  # eager, on the stream of the captures
        plan.run(qs[6], outs[6])
    torch.cuda.synchronize()
    assert torch.equal(outs[6], alone[6])
    for i in range(6):
        for out in outs:
            out.fill_(5.0)
        torch.cuda.synchronize()
        for graph, s in graphs:
            with torch.cuda.stream(s):
                graph.replay()
        plan.run(qs[6], outs[6])
        torch.cuda.synchronize()
        for n, out in enumerate(outs):
            assert torch.equal(out, alone[n]), (i, n)
    assert_parity(outs[0], refs[0], label=f"graphs {config}")


def test_plan_made_in_a_capture_runs_outside_it():
    print("plan made in a capture", flush=True)
    cache, qs, refs = _setup(queries=2)
    plan = None
    out = torch.empty_like(qs[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan = DecodeLaunch(qs[0], cache, config={"split_k": 4}, max_len=max(LENS), total_pages=700)
        plan.run(qs[0], out)
    eager = plan.run(qs[1])  # before the first replay
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert_parity(out, refs[0], label="plan made in a capture")
    assert_parity(eager, refs[1], label="plan made in a capture, eager")
    assert torch.equal(plan.run(qs[1]), eager)


def test_plan_keeps_a_bounded_number_of_streams(monkeypatch):
    print("bounded streams", flush=True)
    monkeypatch.setattr(dec, "_MAX_STREAMS", 3)
    cache, qs, refs = _setup(queries=1)
    plan = DecodeLaunch(qs[0], cache, config={"split_k": 4})
    want = plan.run(qs[0]).clone()
    streams = [torch.cuda.Stream() for _ in range(6)]
    for s in streams + streams[:2]:
        with torch.cuda.stream(s):
            got = plan.run(qs[0])
        s.synchronize()
        assert torch.equal(got, want)
    assert len(plan._states) == 4 and plan._home in plan._states
