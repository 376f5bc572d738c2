"""Decode partitions whose head groups share lines of K and V (several per KV
head, or 64-byte rows of 8-bit caches), which the kernels run on one XCD in an
order of their own: every (sequence, head group, partition) is still computed
once, whatever remains of the grid after the rounds of eight.

Checked bit for bit against the same launch one sequence at a time, and against
the oracle within ``tests/_parity.py``'s tolerance.
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


def _alone(run, q, cache):
    outs = []
    for i in range(len(LENS)):
        c = PagedKVCache(cache.k_cache, cache.v_cache, cache.page_table[i:i + 1].contiguous(),
                         cache.seq_lens[i:i + 1].contiguous(), cache.page_size)
        outs.append(run(q[i:i + 1].contiguous(), c))
    return torch.cat(outs)


@pytest.mark.parametrize("split", [1, 3, 8, 17])
@pytest.mark.parametrize("h,hk,dtype,P", [(12, 1, torch.bfloat16, 1), (10, 2, torch.float32, 16),
                                          (64, 1, torch.float16, 16), (40, 1, torch.float16, 16)])
def test_shared_head_groups(h, hk, dtype, P, split):
    print(f"share H{h}/{hk} {dtype} P{P} split {split}", flush=True)
    k, v, pt, sl = make_paged(LENS, hk, 128, P, dtype, seed=h, device=DEV)
    cache = PagedKVCache(k, v, pt, sl, P)
    q = make_query(len(LENS), h, 128, dtype, seed=h + 1, device=DEV)
    run = lambda q, c: paged_decode_attention(q, c, config={"split_k": split, "num_warps": 4})  # noqa: E731
    out = run(q, cache)
    torch.cuda.synchronize()
    assert torch.equal(out, _alone(run, q, cache))
    ref = ref_attention_paged(q.cpu().float(), k.cpu().float(), v.cpu().float(), pt.cpu(), sl.cpu(), return_fp32=True)
    if dtype == torch.float32:
        assert ((out.cpu() - ref).abs() / ref.abs().clamp_min(1.0)).max().item() <= 1e-5
    else:
        assert_parity(out, ref, label=f"share H{h}/{hk} split {split}")


@pytest.mark.parametrize("split", [1, 3, 8])
@pytest.mark.parametrize("h,hk,d,P", [(8, 8, 64, 16), (6, 2, 64, 16), (8, 2, 64, 1), (3, 3, 64, 32)])
def test_shared_lines_of_8_bit_rows(h, hk, d, P, split):
    print(f"share int8 H{h}/{hk} D{d} P{P} split {split}", flush=True)
    k, v, pt, sl = make_paged(LENS, hk, d, P, torch.float32, seed=h, device="cpu")
    qk, sk = quant_ref.quantize_pages(k, "int8")
    qv, sv = quant_ref.quantize_pages(v, "int8")
    scales = {"k": sk.to(DEV), "v": sv.to(DEV)}
    q = make_query(len(LENS), h, d, torch.float16, seed=h + 1, device=DEV)
    cache = PagedKVCache(qk.to(DEV), qv.to(DEV), pt.to(DEV), sl.to(DEV), P)
    run = lambda q, c: paged_decode_attention_fp8(q, c, scales, config={"split_k": split, "num_warps": 4})  # noqa: E731
    out = run(q, cache)
    torch.cuda.synchronize()
    assert torch.equal(out, _alone(run, q, cache))
    ref = ref_attention_paged(q.cpu(), quant_ref.dequantize_pages(qk, sk, torch.float16),
                              quant_ref.dequantize_pages(qv, sv, torch.float16), pt, sl, return_fp32=True)
    assert_parity(out, ref, label=f"share int8 H{h}/{hk} split {split}")
