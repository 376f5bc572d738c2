"""Balanced decode launches (equal runs of the batch's token blocks, one per
workgroup) against the fp32 oracle: lengths around the 16- to 128-token
blocks, runs that hold many sequences and sequences that many runs share (up
to more than the 64 that one merge step takes), prepared launches whose
lengths change, empty sequences, and a captured launch.

Tolerances: those of ``tests/_parity.py`` (2e-3 before the output's rounding)
and, for fp32, 1e-5 relative to max(1, |ref|): only the order of the fp32 sums
and the exp2 of the scores differ.
"""

from __future__ import annotations

import pytest
import torch

from _parity import assert_parity, make_paged, make_query
from flashattntile_amd import DecodeLaunch, PagedKVCache, paged_decode_attention, paged_decode_attention_fp8
from oracle import quant_ref
from oracle.reference import ref_attention_paged

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [1, 15, 16, 65, 127, 128, 129, 511, 1300]


def _check(out, ref, label):
    if out.dtype == torch.float32:
        rel = ((out.cpu() - ref).abs() / ref.abs().clamp_min(1.0)).max().item()
        assert torch.isfinite(out).all() and rel <= 1e-5, f"{label}: {rel:.3e}"
    else:
        assert_parity(out, ref, label=label)


def _oracle(q, k, v, pt, sl):
    return ref_attention_paged(q.cpu().float(), k.cpu().float(), v.cpu().float(), pt.cpu(), sl.cpu(),
                               return_fp32=True)


@pytest.mark.parametrize("dtype,d,P", [(torch.float16, 128, 16), (torch.bfloat16, 64, 32), (torch.float16, 128, 1),
                                       (torch.bfloat16, 64, 3), (torch.float16, 32, 16), (torch.float32, 32, 7),
                                       (torch.float32, 64, 16), (torch.float32, 128, 16)])
@pytest.mark.parametrize("h,hk", [(8, 2), (6, 1)])
def test_balanced_decode(h, hk, dtype, d, P):
    k, v, pt, sl = make_paged(LENS, hk, d, P, dtype, seed=d + P, device=DEV)
    cache = PagedKVCache(k, v, pt, sl, P)
    q = make_query(len(LENS), h, d, dtype, seed=d, device=DEV)
    ref = _oracle(q, k, v, pt, sl)
    for groups in (1, 2, 5, 200, 1000):  # 1: the library's own number of workgroups
        label = f"balanced {groups} D{d} {dtype} P{P} H{h}/{hk}"
        print(label, flush=True)
        out = paged_decode_attention(q, cache, config={"balanced": groups})
        torch.cuda.synchronize()
        _check(out, ref, label)


@pytest.mark.parametrize("d,P", [(64, 16), (128, 64), (64, 1), (128, 3), (256, 16)])
@pytest.mark.parametrize("mode", ["int8", "float8_e4m3fn"])
def test_balanced_8bit(mode, d, P):
    k, v, pt, sl = make_paged(LENS, 2, d, P, torch.float32, seed=P + 7, device="cpu")
    qk, sk = quant_ref.quantize_pages(k, mode)
    qv, sv = quant_ref.quantize_pages(v, mode)
    q = make_query(len(LENS), 8, d, torch.bfloat16, seed=P + 8, device=DEV)
    cache = PagedKVCache(qk.to(DEV), qv.to(DEV), pt.to(DEV), sl.to(DEV), P)
    ref = ref_attention_paged(q.cpu(), quant_ref.dequantize_pages(qk, sk, torch.bfloat16),
                              quant_ref.dequantize_pages(qv, sv, torch.bfloat16), pt, sl, return_fp32=True)
    for groups in (1, 3, 300):
        label = f"balanced {groups} {mode} D{d} P{P}"
        print(label, flush=True)
        out = paged_decode_attention_fp8(q, cache, {"k": sk.to(DEV), "v": sv.to(DEV)}, config={"balanced": groups})
        torch.cuda.synchronize()
        assert_parity(out, ref, label=label)


@pytest.mark.parametrize("dtype,d,P,batch", [(torch.float16, 128, 16, 300), (torch.float32, 64, 16, 9),
                                             (torch.bfloat16, 64, 1, 1024)])
def test_balanced_plan_follows_the_lengths(dtype, d, P, batch):
    """One prepared launch, other lengths at every run (with empty sequences,
    whose outputs are zero), then captured: the counters are zero again after
    each run.  300 and 1024 sequences: more than one step of the prefix sum."""
    g = torch.Generator().manual_seed(batch)
    lens = torch.randint(1, 400, (batch,), generator=g)
    lens[::7] = 1500 // (1 + batch // 100)
    k, v, pt, sl = make_paged(lens.tolist(), 2, d, P, dtype, seed=batch, device=DEV)
    cache = PagedKVCache(k, v, pt, sl, P)
    q = make_query(batch, 8, d, dtype, seed=3, device=DEV)
    plan = DecodeLaunch(q, cache, config={"balanced": 1})
    out = torch.empty_like(q)
    full = sl.clone()

    def check(run, label):
        for i, cut in enumerate((1.0, 0.37, 0.0, 0.9)):
            sl.copy_((full.double() * cut).to(sl.dtype))
            if cut == 0.9:
                sl[::3] = 0
            print(f"{label} {dtype} B{batch} run {i}", flush=True)
            out.fill_(7.0)
            run()
            torch.cuda.synchronize()
            assert int(plan.counters.abs().max()) == 0
            held = (sl > 0).cpu()
            ref = _oracle(q, k, v, pt, sl.clamp_min(1))
            assert (out[~held.to(DEV)] == 0).all()
            if held.any():
                _check(out[held.to(DEV)], ref[held], f"{label} run {i}")

    check(lambda: plan.run(q, out), "plan")
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        plan.run(q, out)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.run(q, out)
    check(graph.replay, "graph")


@pytest.mark.parametrize("heads", [(32, 1), (4, 4)])
def test_balanced_falls_back(heads):
    """Shapes without a balanced kernel (more than sixteen rows per workgroup,
    more than 1024 sequences) run as partitions."""
    h, hk = heads
    batch = 3 if hk == 1 else 1100
    lens = [1 + (37 * i) % 90 for i in range(batch)]
    k, v, pt, sl = make_paged(lens, hk, 64, 16, torch.float16, seed=11, device=DEV)
    cache = PagedKVCache(k, v, pt, sl, 16)
    q = make_query(batch, h, 64, torch.float16, seed=12, device=DEV)
    ref = _oracle(q, k, v, pt, sl)
    for cfg in ({"balanced": 1}, {"balanced": 1, "num_warps": 8}, {"balanced": 1, "split_k": 2}):
        print(f"balanced fallback H{h}/{hk} {cfg}", flush=True)
        out = paged_decode_attention(q, cache, config=cfg)
        torch.cuda.synchronize()
        _check(out, ref, f"fallback H{h}/{hk} {cfg}")


@pytest.mark.parametrize("dtype,d,P", [(torch.float16, 128, 1), (torch.bfloat16, 64, 3), (torch.float32, 64, 16)])
def test_balanced_plan_takes_unaligned_queries(dtype, d, P):
    """A prepared balanced launch run with contiguous queries that aren't
    16-byte aligned: the generic kernel, in the plan's workspace."""
    k, v, pt, sl = make_paged(LENS, 2, d, P, dtype, seed=31, device=DEV)
    cache = PagedKVCache(k, v, pt, sl, P)
    q = make_query(len(LENS), 8, d, dtype, seed=32, device=DEV)
    ref = _oracle(q, k, v, pt, sl)
    plan = DecodeLaunch(q, cache, config={"balanced": 1, "split_k": 11})
    assert plan._args.balanced
    flat = torch.empty(q.numel() + 16, dtype=dtype, device=DEV)
    for offset in (0, 1, 3, 0):
        label = f"balanced plan, query at {offset} {dtype} D{d} P{P}"
        print(label, flush=True)
        view = flat[offset:offset + q.numel()].view(q.shape)
        view.copy_(q)
        out = plan.run(view)
        torch.cuda.synchronize()
        _check(out, ref, label)
