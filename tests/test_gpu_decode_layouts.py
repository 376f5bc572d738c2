"""Decode over caches whose K/V aren't dense [pages, slots, heads, dim]: K and V
interleaved, head-major pages, padded rows, slots that lie a pool apart, and K
and V of different layouts, on the per-lane, per-load and MFMA kernels, in
partitions (with and without head groups that share lines) and balanced runs.

Checked bit for bit against the dense cache on the same launch (the layout
decides addresses, and in which order head groups run, but no arithmetic), and
against the oracle within ``tests/_parity.py``'s tolerance (fp32: 1e-5 relative
to max(1, |ref|)).
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
LENS = [300, 1, 77, 512, 130, 64, 333]
CONFIGS = [{"split_k": 1}, {"split_k": 3, "num_warps": 4}, {"split_k": 8, "num_warps": 8}, {"balanced": 1},
           {"balanced": 5}]


def _like(x, order, pad=0):
    """``x`` in storage whose axes run in ``order``, rows ``pad`` elements apart."""
    shape = [x.shape[i] for i in order]
    back = [order.index(i) for i in range(4)]
    store = torch.zeros(*shape[:3], shape[3] + pad, dtype=x.dtype, device=x.device)
    out = store[..., :shape[3]].permute(*back)
    out.copy_(x)
    return out


def _layouts(k, v):
    pad = 16 // k.element_size()
    both = torch.stack([k, v], dim=2).contiguous()
    heads = torch.stack([k, v], dim=3).contiguous()
    yield "K and V by token", both[:, :, 0], both[:, :, 1]
    yield "K and V by head", heads[:, :, :, 0], heads[:, :, :, 1]
    yield "head-major pages", _like(k, (0, 2, 1, 3)), _like(v, (0, 2, 1, 3))
    yield "heads outside", _like(k, (2, 0, 1, 3)), _like(v, (2, 0, 1, 3))
    yield "slots outside", _like(k, (1, 0, 2, 3)), _like(v, (1, 0, 2, 3))
    yield "padded rows", _like(k, (0, 1, 2, 3), pad), _like(v, (0, 1, 2, 3), 2 * pad)
    yield "two layouts", k, _like(v, (0, 2, 1, 3), pad)


def _run(label, call, k, v, pt, sl, P, ref):
    dense = PagedKVCache(k, v, pt, sl, P)
    for cfg in CONFIGS:
        want = call(dense, cfg)
        torch.cuda.synchronize()
        if want.dtype == torch.float32:
            assert ((want.cpu() - ref).abs() / ref.abs().clamp_min(1.0)).max().item() <= 1e-5
        else:
            assert_parity(want, ref, label=f"{label} {cfg}")
        for name, kk, vv in _layouts(k, v):
            print(f"{label} {cfg} {name}", flush=True)
            assert torch.equal(kk, k) and torch.equal(vv, v)
            got = call(PagedKVCache(kk, vv, pt, sl, P), cfg)
            torch.cuda.synchronize()
            assert torch.equal(got, want), (label, cfg, name)


@pytest.mark.parametrize("dtype,d,P,h,hk", [(torch.float16, 128, 1, 8, 2), (torch.bfloat16, 64, 3, 6, 2),
                                            (torch.float16, 32, 16, 8, 4), (torch.bfloat16, 256, 16, 8, 2),
                                            (torch.float32, 64, 16, 12, 1), (torch.float32, 32, 7, 4, 4),
                                            (torch.float16, 128, 16, 8, 2), (torch.bfloat16, 64, 32, 12, 3),
                                            (torch.float16, 128, 16, 40, 1)])
def test_layouts(dtype, d, P, h, hk):
    k, v, pt, sl = make_paged(LENS, hk, d, P, dtype, seed=d + P, device=DEV)
    q = make_query(len(LENS), h, d, dtype, seed=d, device=DEV)
    ref = ref_attention_paged(q.cpu().float(), k.cpu().float(), v.cpu().float(), pt.cpu(), sl.cpu(), return_fp32=True)
    _run(f"layouts {dtype} D{d} P{P} H{h}/{hk}", lambda c, cfg: paged_decode_attention(q, c, config=cfg), k, v, pt, sl,
         P, ref)


@pytest.mark.parametrize("mode", ["int8", "float8_e4m3fn"])
@pytest.mark.parametrize("qdtype,d,P,h,hk", [(torch.float16, 64, 1, 8, 2), (torch.bfloat16, 128, 3, 8, 2),
                                             (torch.float16, 256, 16, 4, 4), (torch.bfloat16, 64, 16, 8, 8),
                                             (torch.float16, 128, 16, 8, 2)])
def test_layouts_8bit(qdtype, d, P, h, hk, mode):
    k, v, pt, sl = make_paged(LENS, hk, d, P, torch.float32, seed=d + P, device="cpu")
    qk, sk = quant_ref.quantize_pages(k, mode)
    qv, sv = quant_ref.quantize_pages(v, mode)
    scales = {"k": sk.to(DEV), "v": sv.to(DEV)}
    q = make_query(len(LENS), h, d, qdtype, seed=d, device=DEV)
    ref = ref_attention_paged(q.cpu(), quant_ref.dequantize_pages(qk, sk, qdtype),
                              quant_ref.dequantize_pages(qv, sv, qdtype), pt, sl, return_fp32=True)
    # codes moved as bytes: torch copies no fp8 views
    kb, vb = qk.to(DEV).view(torch.int8), qv.to(DEV).view(torch.int8)

    def call(c, cfg):
        typed = PagedKVCache(c.k_cache.view(qk.dtype), c.v_cache.view(qk.dtype), c.page_table, c.seq_lens, P)
        return paged_decode_attention_fp8(q, typed, scales, config=cfg)

    _run(f"layouts {mode} {qdtype} D{d} P{P} H{h}/{hk}", call, kb, vb, pt.to(DEV), sl.to(DEV), P, ref)
