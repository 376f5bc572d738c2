"""The check kernel (fat_check_begin / fat_check_wait) against the torch
reductions it stands in for, over the forms that the validated calls accept:
strided tables and lengths, negative and empty sequences, tables of one and
of many workgroups, several threads and streams; and that a validated call is
refused under capture."""

from __future__ import annotations

import threading

import pytest
import torch

from flashattntile_amd import PagedKVCache, _hip, prefill_attention
from flashattntile_amd.kernels import prefill as pre
from flashattntile_amd.paging import cache_stats

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _i32(x):
    return torch.tensor(x, dtype=torch.int32)


def _stream():
    return _hip.current_stream_handle(DEV)


def _varlen(cq, ck):
    r = _hip.check_begin(_hip.CHECK_VARLEN, _stream(), DEV, cu_q=cq.to(DEV), cu_k=ck.to(DEV)).wait()
    return [r[3], r[5], r[4], r[6], r[7] & 1, r[7] & 2, r[7] & 4, r[8], r[9], r[10] >= 0, r[10], r[11]]


def _agree(got, want):
    """Same verdicts; the first keyless sequence only where there is one."""
    assert got[:4] == want[:4] and got[7:9] == want[7:9]
    assert [bool(x) for x in got[4:7]] == [bool(x) for x in want[4:7]] and bool(got[9]) == bool(want[9])
    if want[9]:
        assert got[10:] == want[10:]


@pytest.mark.parametrize("B", [1, 2, 63, 257, 1000])
def test_varlen(B):
    print(f"check varlen B{B}", flush=True)
    g = torch.Generator().manual_seed(B)
    for lo in (0, -3):  # decreasing offsets among them
        cq = torch.cat([torch.zeros(1), torch.randint(lo, 50, (B,), generator=g).cumsum(0)]).to(torch.int32)
        ck = torch.cat([torch.ones(1), torch.randint(lo, 50, (B,), generator=g).cumsum(0)]).to(torch.int32)
        _agree(_varlen(cq, ck), pre._varlen_stats(cq, ck))


@pytest.mark.parametrize("B,max_pages,P", [(1, 1, 1), (3, 7, 5), (5, 5000, 1), (64, 1000, 16), (2000, 3, 16)])
def test_cache_and_paged(B, max_pages, P):
    print(f"check paged B{B} pages {max_pages} P{P}", flush=True)
    g = torch.Generator().manual_seed(B)
    wide = torch.randint(-9, 1 << 30, (B, max_pages + 3), generator=g, dtype=torch.int32)
    lens = torch.randint(-2, max_pages * P + 20, (B,), generator=g, dtype=torch.int32)
    cq = torch.cat([torch.zeros(1), torch.randint(-1, 9, (B,), generator=g).cumsum(0)]).to(torch.int32)
    k = torch.zeros(1, P, 1, 16)
    for table in (wide, wide[:, 2:2 + max_pages]):  # dense, strided rows
        cpu = PagedKVCache(k, k, table, lens, P)
        dev = PagedKVCache(k.to(DEV), k.to(DEV), wide.to(DEV)[:, 2:2 + max_pages] if table is not wide else
                           wide.to(DEV), lens.to(DEV), P)
        assert cache_stats(dev, True) == cache_stats(cpu, True)
        r = _hip.check_begin(_hip.CHECK_PAGED, _stream(), DEV, cu_q=cq.to(DEV), seq_lens=dev.seq_lens,
                             page_table=dev.page_table, page_size=P).wait()
        w = pre._paged_stats(cpu, cq)
        assert [r[3], r[4], r[8], r[0], r[1], r[12], r[13]] == [w[0], w[1], w[3], w[5], w[6], w[7], w[8]]
        assert [bool(r[7] & 1), bool(r[7] & 4), r[10] >= 0] == [bool(w[2]), bool(w[4]), bool(w[9])]
        if w[9]:
            assert [r[10], r[11]] == w[10:]


@pytest.mark.parametrize("B,max_pages,P", [(1, 1, 1), (7, 9, 4), (300, 5, 16)])
def test_append_targets(B, max_pages, P):
    print(f"check append B{B}", flush=True)
    g = torch.Generator().manual_seed(B)
    table = torch.randint(-9, 1000, (B, max_pages), generator=g, dtype=torch.int32)
    lens = torch.randint(-2, max_pages * P + 5, (B,), generator=g, dtype=torch.int32)
    r = _hip.check_begin(_hip.CHECK_APPEND, _stream(), DEV, seq_lens=lens.to(DEV), page_table=table.to(DEV),
                         page_size=P).wait()
    block = torch.div(lens, P, rounding_mode="floor").clamp(0, max_pages - 1).long()
    ids = table[torch.arange(B), block]
    assert [r[0], r[1], r[12], r[13]] == [int(x) for x in (lens.min(), lens.max(), ids.min(), ids.max())]


@pytest.mark.parametrize("n", [1, 255, 4097, 300000])
def test_float_range(n):
    print(f"check range {n}", flush=True)
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, generator=g)
    assert _hip.float_range(x.to(DEV)) == (x.min().item(), x.max().item())
    x[n // 2] = -float("inf")
    assert _hip.float_range(x.to(DEV)) == (x.min().item(), x.max().item())
    x[n // 3] = float("nan")
    assert all(v != v for v in _hip.float_range(x.to(DEV)))


def test_threads_and_streams():
    """Each thread has its own words: concurrent checks on several streams
    keep their answers apart."""
    print("check threads", flush=True)
    wrong = []

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream(DEV)):
            for i in range(50):
                n = 100 * k + i
                got = _varlen(_i32([0, n]), _i32([0, n + 1]))
                if got[2:4] != [n, n + 1]:
                    wrong.append((k, i, got))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong[:3]


def test_a_check_left_behind_does_not_reach_the_next_one():
    print("check left behind", flush=True)
    a, b = _i32([0, 5]).to(DEV), _i32([0, 9]).to(DEV)
    _hip.check_begin(_hip.CHECK_VARLEN, _stream(), DEV, cu_q=a, cu_k=a)  # never waited for
    r = _hip.check_begin(_hip.CHECK_VARLEN, _stream(), DEV, cu_q=b, cu_k=b).wait()
    assert r[4] == 9


def test_validated_calls_are_refused_under_capture():
    print("check capture", flush=True)
    q = torch.randn(8, 4, 64, device=DEV, dtype=torch.float16)
    cu = _i32([0, 8]).to(DEV)
    want = prefill_attention(q, q, q, cu, cu, 8, 8)
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream(DEV)
    with torch.cuda.stream(side):
        graph.capture_begin()
        with pytest.raises(RuntimeError, match="capturing"):
            prefill_attention(q, q, q, cu, cu, 8, 8)
        graph.capture_end()
    torch.cuda.synchronize()
    assert torch.equal(prefill_attention(q, q, q, cu, cu, 8, 8), want)


@pytest.mark.parametrize("default", ["cuda", "meta"])
def test_validated_calls_under_a_default_device(default):
    """The page-locked words of a thread's first check, whatever device the
    program has tensors made on by default."""
    from flashattntile_amd import append_tokens, paged_decode_attention, paged_prefill_attention, quantize_cache

    print(f"check under default device {default}", flush=True)
    q = torch.randn(2, 4, 64, device=DEV, dtype=torch.float16)
    pages = torch.randn(4, 16, 2, 64, device=DEV, dtype=torch.float16)
    table = _i32([[0, 1], [2, 3]]).to(DEV)
    cu = _i32([0, 2]).to(DEV)
    cu2 = _i32([0, 1, 2]).to(DEV)

    def cache():
        return PagedKVCache(pages.clone(), pages.clone(), table, _i32([20, 5]).to(DEV), 16)

    def calls(c):
        yield prefill_attention(q, q, q, cu, cu, 2, 2)
        yield paged_decode_attention(q, c)
        yield paged_prefill_attention(q, c, cu2, 1)
        yield quantize_cache(c, "int8")[1].k
        append_tokens(c, pages[:2, 0].contiguous(), pages[:2, 1].contiguous())
        yield c.k_cache

    want = [t.clone() for t in calls(cache())]
    caches = [cache() for _ in want]  # one per call: an error of one doesn't end the others
    got, errors = {}, []

    def run(i):  # a thread's own check and default device
        torch.set_default_device(default)
        try:
            got[i] = [t.clone() for t in calls(caches[i])][i]
        except Exception as exc:
            errors.append((i, exc))

    for i in range(len(want)):
        thread = threading.Thread(target=run, args=(i,))
        thread.start()
        thread.join(60)
    torch.cuda.synchronize()
    assert not errors, errors
    assert all(torch.equal(got[i], want[i]) for i in range(len(want)))
