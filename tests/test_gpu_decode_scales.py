"""8-bit decode on the VALU and MFMA kernels where the table columns past a
sequence's pages name a page that no sequence holds and whose scales are not
finite: one partition, proportional and fixed-size ones, balanced runs and
several tokens per sequence, against the dequantise-then-attend oracle.

Tolerances: ``tests/_parity.py``.
"""

from __future__ import annotations

import pytest
import torch

from _parity import assert_parity, make_paged
from flashattntile_amd import PagedKVCache, paged_decode_attention_fp8, paged_decode_attention_multi
from oracle import quant_ref
from oracle.reference import ref_attention_paged, ref_attention_varlen

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [4, 15, 16, 17, 33, 63, 65, 127, 129, 500]
CONFIGS = [{"split_k": 1}, {"split_k": 3}, {"split_k": 5, "pages_per_split": 3}, {"split_k": 1, "num_warps": 8},
           {"split_k": 3, "kernel": "valu"}, {"split_k": 1, "kernel": "valu", "num_warps": 8}, {"balanced": 3}]


def _inputs(mode, d, P, shape, qdtype):
    k, v, pt, sl = make_paged(LENS, 2, d, P, torch.float32, seed=P + d, device="cpu", extra_pages=1)
    qk, sk = quant_ref.quantize_pages(k, mode)
    qv, sv = quant_ref.quantize_pages(v, mode)
    held = torch.zeros(k.shape[0], dtype=torch.bool)
    for b, n in enumerate(LENS):
        held[pt[b, :-(-n // P)].long()] = True
    spare = int((~held).nonzero()[0])
    for b, n in enumerate(LENS):
        pt[b, -(-n // P):] = spare
    q = torch.randn(shape, generator=torch.Generator().manual_seed(d)).to(qdtype)
    kd, vd = quant_ref.dequantize_pages(qk, sk, qdtype), quant_ref.dequantize_pages(qv, sv, qdtype)
    sk[spare], sv[spare] = float("nan"), float("inf")
    cache = PagedKVCache(qk.to(DEV), qv.to(DEV), pt.to(DEV), sl.to(DEV), P)
    return q, cache, {"k": sk.to(DEV), "v": sv.to(DEV)}, kd, vd


@pytest.mark.parametrize("d,P", [(64, 16), (128, 8), (128, 32)])
@pytest.mark.parametrize("qdtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mode", ["int8", "float8_e4m3fn"])
def test_scales_of_unused_columns(mode, qdtype, d, P):
    q, cache, scales, kd, vd = _inputs(mode, d, P, (len(LENS), 8, d), qdtype)
    ref = ref_attention_paged(q, kd, vd, cache.page_table.cpu(), cache.seq_lens.cpu(), return_fp32=True)
    for cfg in CONFIGS:
        label = f"unused scales {mode} {qdtype} D{d} P{P} {cfg}"
        print(label, flush=True)
        out = paged_decode_attention_fp8(q.to(DEV), cache, scales, config=cfg)
        torch.cuda.synchronize()
        assert_parity(out, ref, label=label)


@pytest.mark.parametrize("mode", ["int8", "float8_e4m3fn"])
def test_scales_of_unused_columns_multi(mode):
    q, cache, scales, kd, vd = _inputs(mode, 128, 16, (len(LENS), 4, 8, 128), torch.float16)
    table = cache.page_table.cpu()
    refs = []
    for b, n in enumerate(LENS):
        ids = table[b, :-(-n // 16)].long()
        rows = [x[ids].reshape(-1, 2, 128)[:n] for x in (kd, vd)]
        refs.append(ref_attention_varlen(q[b], *rows, torch.tensor([0, 4], dtype=torch.int32),
                                         torch.tensor([0, n], dtype=torch.int32), causal=True, return_fp32=True))
    for cfg in ({"split_k": 1}, {"split_k": 3}, {"balanced": 3}):
        label = f"unused scales, four tokens, {mode} {cfg}"
        print(label, flush=True)
        out = paged_decode_attention_multi(q.to(DEV), cache, scales=scales, config=cfg)
        torch.cuda.synchronize()
        assert_parity(out, torch.stack(refs), label=label)
