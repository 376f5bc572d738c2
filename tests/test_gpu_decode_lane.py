"""The per-lane form of the VALU decode (pages that one load can straddle,
fp32 caches, head_dim 32 and 256) against the fp32 oracle, at lengths around
its 16-, 32- and 64-token units, with partitions of fixed and of proportional
size, and beside the generic kernel forced on the same inputs.

Tolerances: those of ``tests/_parity.py`` (2e-3 before the output's rounding)
and, for fp32, 1e-5 relative to max(1, |ref|): only the order of the fp32 sums
and the exp2 of the scores differ.
"""

from __future__ import annotations

import pytest
import torch

from _parity import assert_parity, make_paged, make_query
from flashattntile_amd import PagedKVCache, paged_decode_attention, paged_decode_attention_fp8
from oracle import quant_ref
from oracle.reference import ref_attention_paged

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [1, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129, 500]
# (split_k, pages_per_split): one partition, proportional ones, fixed-size ones
# whose later partitions are empty for the short sequences.
PARTS = [(1, None), (3, None), (5, 40)]


def _check(out, ref, label):
    if out.dtype == torch.float32:
        rel = ((out.cpu() - ref).abs() / ref.abs().clamp_min(1.0)).max().item()
        print(f"{label} max_rel={rel:.3e}", flush=True)
        assert torch.isfinite(out).all() and rel <= 1e-5, f"{label}: {rel:.3e}"
    else:
        assert_parity(out, ref, label=label)


def _config(split, pps, P):
    cfg = {"split_k": split}
    if pps is not None:
        cfg["pages_per_split"] = max(1, pps // P)
    return cfg


@pytest.mark.parametrize("P", [1, 3, 7, 16])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 32), (torch.float16, 64), (torch.bfloat16, 128),
                                     (torch.float16, 256), (torch.bfloat16, 256), (torch.float32, 32),
                                     (torch.float32, 64), (torch.float32, 128)])
@pytest.mark.parametrize("h,hk", [(8, 2), (6, 1)])
def test_lane_decode(h, hk, dtype, d, P):
    k, v, pt, sl = make_paged(LENS, hk, d, P, dtype, seed=d + P, device=DEV)
    cache = PagedKVCache(k, v, pt, sl, P)
    q = make_query(len(LENS), h, d, dtype, seed=d, device=DEV)
    ref = ref_attention_paged(q.cpu().float(), k.cpu().float(), v.cpu().float(), pt.cpu(), sl.cpu(),
                              return_fp32=True)
    for split, pps in PARTS:
        for waves in (4, 8):
            cfg = {**_config(split, pps, P), "num_warps": waves}
            label = f"lane D{d} {dtype} P{P} {cfg}"
            print(label, flush=True)
            out = paged_decode_attention(q, cache, config=cfg)
            torch.cuda.synchronize()
            _check(out, ref, label)
    gen = paged_decode_attention(q, cache, config={"split_k": 3, "kernel": "generic"})
    torch.cuda.synchronize()
    _check(gen, ref, f"generic D{d} {dtype} P{P}")


@pytest.mark.parametrize("d,P", [(64, 1), (128, 3), (256, 5), (256, 16)])
@pytest.mark.parametrize("qdtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mode", ["int8", "float8_e4m3fn"])
def test_lane_decode_8bit(mode, qdtype, d, P):
    k, v, pt, sl = make_paged(LENS, 2, d, P, torch.float32, seed=P + 7, device="cpu")
    qk, sk = quant_ref.quantize_pages(k, mode)
    qv, sv = quant_ref.quantize_pages(v, mode)
    q = make_query(len(LENS), 8, d, qdtype, seed=P + 8, device=DEV)
    cache = PagedKVCache(qk.to(DEV), qv.to(DEV), pt.to(DEV), sl.to(DEV), P)
    ref = ref_attention_paged(q.cpu(), quant_ref.dequantize_pages(qk, sk, qdtype),
                              quant_ref.dequantize_pages(qv, sv, qdtype), pt, sl, return_fp32=True)
    for split, pps in PARTS:
        label = f"lane {mode} {qdtype} D{d} P{P} split {split}"
        print(label, flush=True)
        out = paged_decode_attention_fp8(q, cache, {"k": sk.to(DEV), "v": sv.to(DEV)}, config=_config(split, pps, P))
        torch.cuda.synchronize()
        assert_parity(out, ref, label=label)


def test_unaligned_queries_keep_the_generic_kernel():
    """A query view whose rows are not 16-byte aligned, which the generic
    kernel reads element by element."""
    print("lane unaligned q", flush=True)
    k, v, pt, sl = make_paged([40, 70], 2, 128, 1, torch.float16, seed=3, device=DEV)
    wide = make_query(2, 8, 128 + 2, torch.float16, seed=4, device=DEV)
    from flashattntile_amd.kernels.decode import paged_decode_launch

    q = wide[:, :, 1:129]
    assert q.data_ptr() % 16 and not q.is_contiguous()
    out = paged_decode_launch(q, PagedKVCache(k, v, pt, sl, 1), 128 ** -0.5, 1, out=torch.empty_like(q))
    torch.cuda.synchronize()
    ref = ref_attention_paged(q.cpu().float(), k.cpu().float(), v.cpu().float(), pt.cpu(), sl.cpu(),
                              return_fp32=True)
    assert_parity(out, ref, label="lane unaligned q")


@pytest.mark.parametrize("d,P", [(64, 1), (128, 3), (256, 16)])
@pytest.mark.parametrize("qdtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mode", ["int8", "float8_e4m3fn"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_lane_scales_of_unused_columns(mode, qdtype, d, P, bad):
    """Table columns past a sequence's pages name a page that no sequence
    holds and whose scales are not finite."""
    k, v, pt, sl = make_paged(LENS, 2, d, P, torch.float32, seed=P + 7, device="cpu", extra_pages=1)
    qk, sk = quant_ref.quantize_pages(k, mode)
    qv, sv = quant_ref.quantize_pages(v, mode)
    held = torch.zeros(k.shape[0], dtype=torch.bool)
    for b, n in enumerate(LENS):
        held[pt[b, :-(-n // P)].long()] = True
    spare = int((~held).nonzero()[0])
    for b, n in enumerate(LENS):
        pt[b, -(-n // P):] = spare
    q = make_query(len(LENS), 8, d, qdtype, seed=P + 8, device=DEV)
    ref = ref_attention_paged(q.cpu(), quant_ref.dequantize_pages(qk, sk, qdtype),
                              quant_ref.dequantize_pages(qv, sv, qdtype), pt, sl, return_fp32=True)
    sk[spare], sv[spare] = bad, bad
    cache = PagedKVCache(qk.to(DEV), qv.to(DEV), pt.to(DEV), sl.to(DEV), P)
    for cfg in [{**_config(split, pps, P), "num_warps": w} for split, pps in PARTS for w in (4, 8)] + [{"balanced": 3}]:
        label = f"lane {mode} {qdtype} D{d} P{P} {cfg}, scales of {bad} past the end"
        print(label, flush=True)
        out = paged_decode_attention_fp8(q, cache, {"k": sk.to(DEV), "v": sv.to(DEV)}, config=cfg)
        torch.cuda.synchronize()
        assert_parity(out, ref, label=label)


def _hide(q, k, pt, P, spans):
    """Scores of -inf for the tokens of ``spans`` (per sequence): dim 0 of their
    K is -inf, and that of every query is positive."""
    q[..., 0] = q[..., 0].abs() + 0.5
    for b, (lo, hi) in spans:
        for t in range(lo, hi):
            k[int(pt[b, t // P]), t % P, :, 0] = -float("inf")


@pytest.mark.parametrize("P", [1, 3, 16])
@pytest.mark.parametrize("dtype,d", [(torch.float16, 32), (torch.float16, 128), (torch.bfloat16, 64),
                                     (torch.bfloat16, 256), (torch.float32, 64)])
def test_units_of_minus_infinity(dtype, d, P):
    """Whole units, waves and partitions whose scores are -inf beside others
    that are not, as the generic kernel takes them (its 32-token tiles hold
    finite scores first)."""
    lens = [600, 130, 700]
    k, v, pt, sl = make_paged(lens, 2, d, P, dtype, seed=d + P, device="cpu", poison=False)
    q = make_query(len(lens), 8, d, dtype, seed=d, device="cpu")
    _hide(q, k, pt, P, [(0, (64, 320)), (1, (32, 128)), (2, (256, 700))])
    ref = ref_attention_paged(q.float(), k.float(), v.float(), pt, sl, return_fp32=True)
    assert torch.isfinite(ref).all()
    cache = PagedKVCache(k.to(DEV), v.to(DEV), pt.to(DEV), sl.to(DEV), P)
    for cfg in ({"split_k": 1, "num_warps": 4}, {"split_k": 1, "num_warps": 8}, {"split_k": 3}, {"split_k": 20},
                {"balanced": 4}, {"split_k": 1, "kernel": "generic"}):
        label = f"-inf units D{d} {dtype} P{P} {cfg}"
        print(label, flush=True)
        out = paged_decode_attention(q.to(DEV), cache, config=cfg)
        torch.cuda.synchronize()
        _check(out, ref, label)
