"""Packed fp32 prefill on the fp32 matrix instructions (csrc/prefill_f32.hip)
against the fp32 oracle, at lengths around its 32-row blocks, 32-key tiles and
the 128 keys that its four waves take between them, and against 64-bit
arithmetic beside the generic VALU kernel.

Tolerance against the oracle: 1e-5 relative to max(1, |ref|), as for the
generic kernel (only the order of the fp32 sums and exp2 differ).
"""

from __future__ import annotations

import pytest
import torch

from flashattntile_amd import prefill_attention
from flashattntile_amd.kernels.prefill import prefill_launch
from oracle.reference import ref_attention_varlen

pytestmark = pytest.mark.gpu
DEV = "cuda"
RTOL = 1e-5


def _case(lq, lk, h, hk, d, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(sum(lq), h, d, generator=g).to(DEV)
    k = torch.randn(sum(lk), hk, d, generator=g).to(DEV)
    v = torch.randn(sum(lk), hk, d, generator=g).to(DEV)
    cu = [torch.tensor([0] + torch.tensor(x).cumsum(0).tolist(), dtype=torch.int32, device=DEV) for x in (lq, lk)]
    return q, k, v, cu[0], cu[1]


def _check(out, q, k, v, cq, ck, causal, label, scale=None):
    ref = ref_attention_varlen(q.cpu(), k.cpu(), v.cpu(), cq.cpu(), ck.cpu(), causal=causal, softmax_scale=scale)
    rel = ((out.cpu() - ref).abs() / ref.abs().clamp_min(1.0)).max().item()
    print(f"{label} max_rel={rel:.3e}", flush=True)
    assert torch.isfinite(out).all() and rel <= RTOL, f"{label}: {rel:.3e}"


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("h,hk", [(4, 4), (8, 2), (3, 1)])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_f32_prefill(d, h, hk, causal):
    lq = [1, 31, 32, 33, 64, 65, 0, 100, 129, 300]
    lk = [1, 31, 32, 33, 64, 65, 0, 100, 129, 300]
    label = f"f32 prefill D{d} H{h}/{hk} causal={causal}"
    print(label, flush=True)
    args = _case(lq, lk, h, hk, d, seed=d + h)
    out = prefill_attention(*args, max(lq), max(lk), causal=causal)
    torch.cuda.synchronize()
    _check(out, *args, causal, label)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("scale", [None, -0.1, 0.0])
def test_f32_prefill_chunks_and_scales(d, scale):
    """More keys than queries (tiles that no row of a wave sees), odd scales."""
    lq, lk = [1, 5, 40, 33, 7], [500, 128, 129, 1000, 7]
    label = f"f32 prefill chunks D{d} scale={scale}"
    print(label, flush=True)
    args = _case(lq, lk, 4, 2, d, seed=d)
    out = prefill_attention(*args, max(lq), max(lk), causal=True, softmax_scale=scale)
    torch.cuda.synchronize()
    _check(out, *args, True, label, scale)


@pytest.mark.parametrize("d", [32, 128])
def test_f32_prefill_output_rows_8_byte_aligned(d):
    lq = [50, 3]
    q, k, v, cq, ck = _case(lq, lq, 4, 2, d, seed=9)
    wide = torch.full((53, 4, d + 2), 7.0, device=DEV)
    out = wide[:, :, :d]
    print(f"f32 prefill 8-byte rows D{d}", flush=True)
    prefill_launch(q, k, v, cq, ck, 50, 50, True, d ** -0.5, out=out)
    torch.cuda.synchronize()
    _check(out, q, k, v, cq, ck, True, f"f32 prefill 8-byte rows D{d}")
    assert (wide[:, :, d:] == 7.0).all()


@pytest.mark.parametrize("d", [64, 128])
def test_f32_prefill_no_further_from_64_bits_than_the_generic_kernel(d):
    """2-norm error against float64, within 1.2 x the VALU kernel's (two
    summation orders of the same length differ by less)."""
    lq = [777]
    q, k, v, cq, ck = _case(lq, lq, 4, 2, d, seed=d + 1)
    print(f"f32 prefill error D{d}", flush=True)
    outs = [prefill_attention(q, k, v, cq, ck, 777, 777, config=c) for c in (None, {"kernel": "generic"})]
    torch.cuda.synchronize()
    mask = torch.ones(777, 777, dtype=torch.bool, device=DEV).triu(1)
    errs = [0.0, 0.0]
    for hh in range(4):
        s = (q[:, hh].double() * d ** -0.5) @ k[:, hh // 2].double().t()
        ref = torch.softmax(s.masked_fill(mask, float("-inf")), -1) @ v[:, hh // 2].double()
        for i, o in enumerate(outs):
            errs[i] += (o[:, hh].double() - ref).square().sum().item() / ref.square().sum().item()
    print(f"matrix {errs[0] ** 0.5:.3e} valu {errs[1] ** 0.5:.3e}", flush=True)
    assert errs[0] ** 0.5 <= 1.2 * errs[1] ** 0.5


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_f32_prefill_infinite_scores(d, causal):
    """Tiles whose scores are all -inf (the first, one wave's every tile), a
    row that sees nothing else (zeros), and scores of +inf (NaN), beside the
    generic kernel on the same inputs."""
    print(f"f32 prefill infinite scores D{d} causal={causal}", flush=True)
    lens = [300, 200]
    q, k, v, cq, ck = _case(lens, lens, 4, 2, d, seed=d)
    q[..., 0] = q[..., 0].abs() + 0.5
    k[0:32, :, 0] = -float("inf")  # the first tile of sequence 0
    k[160:192, :, 0] = -float("inf")
    for t in range(1, 6, 4):  # the tiles that one wave takes of sequence 1
        k[300 + 32 * t:300 + min(32 * t + 32, 200), :, 0] = -float("inf")
    args = (q, k, v, cq, ck)
    out = prefill_attention(*args, max(lens), max(lens), causal=causal)
    gen = prefill_attention(*args, max(lens), max(lens), causal=causal, config={"kernel": "generic"})
    torch.cuda.synchronize()
    if causal:  # rows 0 - 31 of sequence 0 see only hidden keys
        assert (out[:32] == 0).all() and (gen[:32] == 0).all()
    ref = ref_attention_varlen(q.cpu(), k.cpu(), v.cpu(), cq.cpu(), ck.cpu(), causal=causal)
    for got in (out, gen):
        seen = slice(32 if causal else 0, None)
        rel = ((got.cpu() - ref).abs() / ref.abs().clamp_min(1.0))[seen].max().item()
        assert torch.isfinite(got).all() and rel <= RTOL, rel
    k[100, :, 0] = float("inf")
    out = prefill_attention(*args, max(lens), max(lens), causal=causal)
    gen = prefill_attention(*args, max(lens), max(lens), causal=causal, config={"kernel": "generic"})
    torch.cuda.synchronize()
    assert torch.equal(out.isnan(), gen.isnan()) and out[100:300].isnan().all() and not out[300:].isnan().any()
    assert out[:100].isnan().any() != causal
