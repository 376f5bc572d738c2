"""A prepared decode launch's workspace covers the form that each of its runs
takes, whatever the query's address, and the library refuses a launch that
would write past the workspace it was told of (no kernel runs here)."""

from __future__ import annotations

import ctypes
import itertools
import re

import pytest
import torch

from flashattntile_amd import _hip
from flashattntile_amd.kernels.decode import DEFAULT_CONFIG, _plan_workspace_bytes


def _written(a) -> int:
    """Bytes of workspace that a launch of ``a`` writes, as its refusal of a
    workspace of one byte names them."""
    a.workspace_bytes = 1
    assert _hip.lib().fat_paged_decode(ctypes.byref(a), None) == 1
    found = re.search(r"needs (\d+) bytes of workspace, the caller's holds 1", _hip.lib().fat_last_error().decode())
    assert found, _hip.lib().fat_last_error()
    return int(found.group(1))


def _block(batch, heads, kv_heads, dim, page, q_dtype, kv_dtype, split_k, tokens=1):
    """A block that passes the library's checks, with addresses that nothing reads."""
    q = torch.empty(batch, tokens, heads, dim, dtype=q_dtype)
    cache = torch.empty(4, page, kv_heads, dim, dtype=kv_dtype)
    scale = torch.empty(4, kv_heads) if kv_dtype.itemsize == 1 else None
    table, lens = torch.zeros(batch, 4, dtype=torch.int32), torch.zeros(batch, dtype=torch.int32)
    if tokens == 1:
        q = q[:, 0]
    a = _hip.decode_args(q, cache, cache, table, lens, q, page, 1.0, split_k, k_scale=scale, v_scale=scale)
    a.q, a.k_cache, a.v_cache = 0x10000, 0x20000, 0x30000
    a.workspace, a.merge_counters = 0x40000, 0x50000
    return a


SHAPES = [
    # batch, heads, kv_heads, dim, page, q, cache, tokens
    (32, 32, 8, 128, 1, torch.float16, torch.float16, 1),
    (64, 64, 8, 128, 3, torch.bfloat16, torch.bfloat16, 1),
    (3, 8, 8, 32, 16, torch.float16, torch.float16, 1),
    (40, 32, 1, 64, 7, torch.float16, torch.int8, 1),
    (5, 16, 2, 256, 16, torch.bfloat16, torch.float8_e4m3fn, 1),
    (32, 32, 8, 64, 16, torch.float32, torch.float32, 1),
    (2000, 8, 8, 128, 16, torch.float32, torch.float32, 1),
]
FAST = [(32, 32, 8, 128, 16, torch.float16, torch.float16, 1), (64, 32, 8, 128, 16, torch.bfloat16, torch.int8, 1),
        (16, 32, 8, 128, 16, torch.float16, torch.float8_e4m3fn, 4), (7, 32, 1, 64, 16, torch.bfloat16,
                                                                    torch.bfloat16, 1)]


@pytest.mark.parametrize("shape", SHAPES + FAST)
@pytest.mark.parametrize("split,balanced", [(1, 1), (2, 1), (11, 1), (64, 1), (11, 300), (11, 4096), (5, 0)])
def test_plan_workspace_covers_every_query_address(shape, split, balanced):
    batch, heads, kv_heads, dim, page, q_dtype, kv_dtype, tokens = shape
    cfg = {**DEFAULT_CONFIG, "split_k": split, "balanced": balanced, "pages_per_split": 0}
    # built on an aligned and on an unaligned query, run on either
    for built, run in itertools.product((0, 2, 4, 8), repeat=2):
        step = q_dtype.itemsize
        if built % step or run % step or ((built or run) and shape in FAST):
            continue  # the other kernels refuse unaligned queries
        a = _block(batch, heads, kv_heads, dim, page, q_dtype, kv_dtype, split, tokens)
        a.q += built
        held = _plan_workspace_bytes(a, cfg)
        a.q += run - built
        if split > 1 or (a.balanced and _hip.decode_balanced_workspace_bytes(a)):
            assert _written(a) <= held, (built, run)


def test_stated_workspace_is_not_exceeded():
    a = _block(32, 32, 8, 128, 1, torch.float16, torch.float16, 11)
    a.balanced = 1
    aligned = _written(a)
    assert aligned == _hip.decode_balanced_workspace_bytes(a)
    a.q += 2  # the generic kernel's partitions
    assert _written(a) == _hip.decode_workspace_bytes(32, 32, 128, 11) > aligned
    a.workspace_bytes = aligned
    assert _hip.lib().fat_paged_decode(ctypes.byref(a), None) == 1
    a.workspace_bytes = -1
    assert _hip.lib().fat_paged_decode(ctypes.byref(a), None) == 1
    assert "workspace_bytes" in _hip.lib().fat_last_error().decode()


@pytest.mark.parametrize("split", [1, 2, 7, 64])
def test_launch_sizes_its_partitions_as_the_library_does(split, monkeypatch):
    from flashattntile_amd.kernels import decode as dec

    seen = []
    monkeypatch.setattr(_hip, "decode_with_args", lambda a, stream: seen.append((a.workspace, a.workspace_bytes)))
    monkeypatch.setattr(_hip, "current_stream_handle", lambda device: 0)
    for shape in ((3, 8, 128), (2, 5, 4, 64)):
        q = torch.empty(*shape)
        rows = shape[0] * (shape[1] if len(shape) == 4 else 1)
        need = _hip.decode_workspace_bytes(rows, shape[-2], shape[-1], split)
        dec._launch_block(_hip.DecodeArgs(), q, split)
        held = torch.empty(max(1, need), dtype=torch.uint8)
        dec._launch_block(_hip.DecodeArgs(), q, split, workspace=held)
        assert [b for _, b in seen] == [need, need] and (split == 1 or seen[1][0] == held.data_ptr())
        seen.clear()
