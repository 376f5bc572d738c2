"""Paged prefill of chunks after long contexts on the wide kernel, K (and fp16
V) read through the page table and bf16 V converted to fp16 first: against the
fp32 oracle and the paged ping-pong kernel, at pages of one, two and more tile
halves, with contexts that end inside a tile, partly filled query blocks, a
sequence's first chunk, garbage past every sequence's end, and magnitudes of V
that fp16 can't hold.

Tolerances: ``tests/_parity.py`` (2e-3 against the oracle, twice that between
two kernels), relative to the largest |V| where that exceeds 1.
"""

from __future__ import annotations

import pytest
import torch

from _parity import assert_parity
from flashattntile_amd import _hip, paged_prefill_attention
from test_gpu_prefill_paged import _case, _ref32

pytestmark = pytest.mark.gpu

# (kv_len, q_len): 160 blocks of the wide kernel at 32 heads, 320 of the ping-pong kernel's.
SHORT = [(3840, 512), (3701, 512), (430, 430), (1999, 512), (701, 500)]
# More sequences than the kernel ranks, two blocks per sequence, the first of them partly filled (6 heads: 204
# blocks, 408 of the ping-pong kernel's).
LONG = [(6000 - 97 * i, 1024 - 11 * i) for i in range(17)]


def _launch(lens, h, hk, P, dtype, seed):
    lens_k, lens_q = [c[0] for c in lens], [c[1] for c in lens]
    q, cache, cu = _case(lens_k, lens_q, h, hk, 128, P, dtype, seed=seed)
    return q, cache, cu, max(lens_q)


def _v_bytes(q, cache, cu, mq, causal, P):
    a = _hip.prefill_paged_args(q, cache.k_cache, cache.v_cache, cache.page_table, cache.seq_lens, cu, q, P, mq,
                                causal, 128 ** -0.5)
    assert _hip.prefill_paged_v_bytes(a) == 0  # the contexts' lengths are not known: the paged kernels
    a.total_k = int(cache.seq_lens.sum())
    need = _hip.prefill_paged_v_bytes(a)
    # fp16 takes the wide kernel wherever bf16 does (which also needs room for
    # its copy of V), and has no workspace to show it by
    a.dtype = _hip.DT_BF16
    assert _hip.prefill_paged_v_bytes(a) > 0
    return need


@pytest.mark.parametrize("P", [16, 32, 256])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_wide_paged_prefill_matches_oracle(dtype, causal, P):
    label = f"wide paged prefill {dtype} P{P} causal={causal}"
    print(label, flush=True)
    q, cache, cu, mq = _launch(SHORT, 32, 8, P, dtype, seed=P)
    assert (_v_bytes(q, cache, cu, mq, causal, P) > 0) == (dtype == torch.bfloat16)
    out = paged_prefill_attention(q, cache, cu, mq, causal=causal)
    pp = paged_prefill_attention(q, cache, cu, mq, causal=causal, config={"kernel": "pingpong"})
    torch.cuda.synchronize()
    assert_parity(out, _ref32(q, cache, cu, causal), label=label)
    assert_parity(out, pp.float().cpu(), tol=4e-3, label=label + " vs ping-pong")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_wide_paged_prefill_more_sequences(dtype):
    label = f"wide paged prefill of 17 {dtype}"
    print(label, flush=True)
    q, cache, cu, mq = _launch(LONG, 6, 2, 16, dtype, seed=17)
    assert (_v_bytes(q, cache, cu, mq, True, 16) > 0) == (dtype == torch.bfloat16)
    out = paged_prefill_attention(q, cache, cu, mq, causal=True)
    pp = paged_prefill_attention(q, cache, cu, mq, causal=True, config={"kernel": "pingpong"})
    torch.cuda.synchronize()
    assert not torch.equal(out, pp)  # two kernels: other tiles, other maxima
    assert_parity(out, _ref32(q, cache, cu, True), label=label)
    assert_parity(out, pp.float().cpu(), tol=4e-3, label=label + " vs ping-pong")


@pytest.mark.parametrize("scale", [-0.05, 0.0])
def test_wide_paged_prefill_large_v_and_scales(scale):
    """bf16 V beyond fp16's range in one (sequence, head) only, under a
    negative and a zero softmax scale."""
    print(f"wide paged prefill large V scale {scale}", flush=True)
    q, cache, cu, mq = _launch(SHORT, 32, 8, 16, torch.bfloat16, seed=5)
    page = int(cache.page_table[1, 3])
    cache.v_cache[page, 2, 4, 7] = 3e5
    out = paged_prefill_attention(q, cache, cu, mq, softmax_scale=scale, causal=True)
    pp = paged_prefill_attention(q, cache, cu, mq, softmax_scale=scale, causal=True, config={"kernel": "pingpong"})
    torch.cuda.synchronize()
    ref = pp.float().cpu()
    lo, hi = int(cu[1]), int(cu[2])
    big = torch.zeros(ref.shape, dtype=torch.bool)
    big[lo:hi, 16:20, 7] = True  # KV head 4 serves query heads 16-19
    assert_parity(torch.where(big, 0.0, out.float().cpu()).to(out.dtype), torch.where(big, 0.0, ref), tol=4e-3,
                  label="large V, other elements")
    rel = ((out.float().cpu() - ref).abs() / ref.abs().clamp_min(1.0))[big].max().item()
    assert rel <= 2 * 2 ** -8 + 4e-3, rel  # two bf16 roundings


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_wide_paged_prefill_first_tile_of_minus_infinity(dtype, causal):
    """A sequence whose first 32 keys, the wide kernel's first tile, all have
    scores of -inf (the ping-pong kernel's first tile holds 64)."""
    label = f"wide paged prefill -inf first tile {dtype} causal={causal}"
    print(label, flush=True)
    q, cache, cu, mq = _launch(SHORT, 32, 8, 16, dtype, seed=9)
    q[..., 0] = q[..., 0].abs() + 0.5
    for b in (0, 3):
        cache.k_cache[cache.page_table[b, :2].long(), :, :, 0] = -float("inf")
    out = paged_prefill_attention(q, cache, cu, mq, causal=causal)
    pp = paged_prefill_attention(q, cache, cu, mq, causal=causal, config={"kernel": "pingpong"})
    torch.cuda.synchronize()
    assert_parity(out, _ref32(q, cache, cu, causal), label=label)
    assert_parity(out, pp.float().cpu(), tol=4e-3, label=label + " vs ping-pong")
