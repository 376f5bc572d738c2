"""Paged decode on MI355X: host side of the HIP kernels in ``csrc/decode.hip``.

Public functions keep the reference signatures and validation
(``flashattn_tile/kernels/decode.py:474-704``):

* :func:`paged_decode_attention` (fp16/bf16 cache, ``decode.py:533``);
* :func:`paged_decode_attention_fp8` (int8 / float8_e4m3fn cache with
  per-(page, KV-head) scales, ``decode.py:645``);

plus :func:`paged_decode_attention_multi`, the multi-token (speculative)
decode the reference lacks (its decode takes one query per sequence,
``decode.py:548-553``).

Differences, all deliberate:

* there is no CPU or Triton fallback: non-ROCm tensors, or a dtype the HIP
  kernels do not take, raise instead of silently running the fp32 reference
  (the oracle lives outside the product, under ``oracle/``);
* the quantised path supports split-K as well;
* ``config=None`` takes the launch stored for this shape in the gfx950
  tuned-config store (:func:`flashattntile_amd.autotune.best_config`, keyed by
  :func:`~flashattntile_amd.autotune.decode_signature`) and otherwise the
  MI355X heuristics: balanced runs
  (:func:`~flashattntile_amd.autotune.decode_balanced`) or partitions
  (:func:`~flashattntile_amd.autotune.decode_split`); an explicit ``split_k``
  is honoured exactly;
* validation costs one check launch that the host polls while it prepares the
  decode, instead of ~6 device->host synchronisations.

:func:`paged_decode_launch` is the sync-free entry below the validation, for
callers (benchmarks, CUDA-graph-style capture loops) that validated once.
"""

from __future__ import annotations

import contextlib
import threading
import warnings

import torch

from .. import _hip
from ..autotune import (best_config, decode_balanced, decode_partition, decode_signature, decode_split,
                        is_ragged)
from ..paging import PagedKVCache, _check_layout, cache_stats

__all__ = [
    "DEFAULT_CONFIG",
    "paged_decode_attention",
    "paged_decode_attention_fp8",
    "paged_decode_attention_multi",
    "paged_decode_launch",
    "resolve_decode_config",
    "DecodeLaunch",
]

# split_k None -> MI355X partition heuristic (split_k and pages_per_split from
# the batch's lengths); an explicit split_k keeps the reference's partitioning
# (ceil(pages / split_k) per sequence) unless pages_per_split is also given.
# num_warps is the number of 64-lane waves per workgroup (4 or 8; None lets the
# library choose from the grid size); num_stages is accepted for signature
# compatibility with the reference's Triton knob and validated the same way,
# but the HIP kernel's pipeline depth is fixed (one 16-token unit prefetched
# per wave).  kernel None lets the library choose the kernel family; "valu",
# "mfma" or "generic" forces one (what a tuning run stores for its shape; the
# generic kernel is the library's own choice only for the shapes the VALU
# kernel's per-lane form does not take either: head_dim 16 and 512, fp32 at
# head_dim 256, 8-bit caches at head_dim 32, unaligned queries).
# balanced: 1 cuts the batch's work into equal runs, one per workgroup, in
# place of split_k partitions per sequence, where the kernel has that form (n >
# 1: with n workgroups; always of 4 waves), 0 doesn't; None: when split_k is None too, by
# :func:`~flashattntile_amd.autotune.decode_balanced`.
DEFAULT_CONFIG = {"split_k": None, "num_warps": None, "num_stages": 2, "pages_per_split": None, "kernel": None,
                  "balanced": None}

_KERNEL_CODES = {None: _hip.KERNEL_AUTO, "valu": _hip.KERNEL_DECODE_VALU, "mfma": _hip.KERNEL_DECODE_MFMA,
                 "generic": _hip.KERNEL_DECODE_GENERIC}

# Element types the HIP decode kernels take for q (and for a cache of the same
# type); int8 / float8_e4m3fn caches take fp16 / bf16 queries.
_DECODE_DTYPES = (torch.float16, torch.bfloat16, torch.float32)

_NO_PAGE = torch.iinfo(torch.int32).max  # the check's page range when no column is used

_QUANT_DTYPES = tuple(d for d in (torch.int8, getattr(torch, "float8_e4m3fn", None)) if d is not None)


def _resolve_config(config: dict | None, q: torch.Tensor, cache: PagedKVCache, max_len: int,
                    total_pages: int, q_len: int = 1) -> dict:
    """``decode.py:474-500``: an explicit config, else the stored winner for
    this shape, else the heuristic.  A stored entry the checks below reject
    is ignored with a warning.  Needs no device synchronisation."""
    if config is None:
        sig = decode_signature(int(q.shape[0]), int(q.shape[-2]), cache.num_kv_heads, cache.head_dim,
                               cache.page_size, max_len, total_pages, cache.k_cache.dtype, q_len)
        stored = best_config("decode", sig)
        if stored:
            try:
                return _merge_config({k: v for k, v in stored.items() if k in DEFAULT_CONFIG}, q, cache, max_len,
                                     total_pages, q_len)
            except ValueError as exc:
                warnings.warn(f"ignoring the stored decode config for {sig}: {exc}", RuntimeWarning, stacklevel=3)
        return _merge_config({}, q, cache, max_len, total_pages, q_len)
    unknown = set(config) - set(DEFAULT_CONFIG)
    if unknown:
        raise ValueError(f"unknown decode config keys: {sorted(unknown)}")
    return _merge_config(config, q, cache, max_len, total_pages, q_len)


def resolve_decode_config(q: torch.Tensor, cache: PagedKVCache, max_len: int, total_pages: int,
                          config: dict | None = None, q_len: int = 1) -> dict:
    """The launch the decode wrappers make for these inputs: ``config`` if
    given, else the stored winner for the shape, else the heuristic.  Host
    work only; ``max_len`` and ``total_pages`` are the batch's longest
    sequence and its page count.  For callers of :func:`paged_decode_launch`
    (benchmarks, capture loops) that validated once."""
    return _resolve_config(config, q, cache, max_len, total_pages, q_len)


def _work_items(q: torch.Tensor, cache: PagedKVCache, kernel: str | None, q_len: int) \
        -> tuple[int, int, bool, bool, bool]:
    """``(rows, items, mfma, shared, balances)`` of a decode launch: the (query head,
    token) rows of one workgroup, the (sequence, head group) pairs of the
    batch, whether the library takes the MFMA kernel (``fat_paged_decode``),
    whether head groups share lines of K and V, which partitions keep on one
    XCD and balanced runs do not (27 sequences of 8167-20782 tokens on an int8
    cache at head_dim 64: 97 us in five partitions, 132 balanced), and whether
    the launch has a balanced form that gains."""
    group = int(q.shape[-2]) // cache.num_kv_heads
    rows = group * q_len
    quantized = cache.k_cache.dtype in _QUANT_DTYPES
    d, page = cache.head_dim, cache.page_size
    per_load = (4 if d == 128 else 8) * (2 if quantized else 1)  # rows that one 16-byte load per lane covers
    fast = q.dtype != torch.float32 and d in (64, 128) and page >= per_load and page & (page - 1) == 0
    if fast:
        per_wg = 32 if kernel == "mfma" or (kernel is None and (quantized or group >= 8)) or q_len > 1 else \
            (8 if group >= 8 else 4)
        balances = quantized if per_wg == 32 else per_wg == 4
    else:  # the per-lane form, else the generic kernel
        per_wg = 4
        balances = d >= (64 if quantized else 32) and d <= (256 if quantized else 128)
    if kernel == "generic":
        per_wg, balances = 8, False
    per_line = 128 // (cache.k_cache.element_size() * d)
    shared = rows > per_wg or (per_line > 1 and cache.num_kv_heads % per_line == 0 and
                               cache.k_cache.stride(2) == cache.v_cache.stride(2) == d)
    items = int(q.shape[0]) * cache.num_kv_heads * -(-rows // per_wg)
    return min(rows, per_wg), items, per_wg == 32, shared, balances and not shared


def _merge_config(config: dict, q: torch.Tensor, cache: PagedKVCache, max_len: int, total_pages: int,
                  q_len: int) -> dict:
    resolved = dict(DEFAULT_CONFIG)
    resolved.update(config)
    waves = resolved["num_warps"]
    if resolved["split_k"] is None:
        batch, heads, hkv, page = int(q.shape[0]), int(q.shape[-2]), cache.num_kv_heads, cache.page_size
        max_pages = -(-max_len // page)
        k = cache.k_cache
        rows, items, mfma, shared, balances = _work_items(q, cache, resolved["kernel"], q_len)
        mean_len = min(max_len, total_pages * page / max(1, batch))
        token_bytes = 2 * cache.head_dim * k.element_size()
        if resolved["balanced"] is None and resolved["pages_per_split"] is None and waves in (None, 4) \
                and balances:
            resolved["balanced"] = int(decode_balanced(max_len, mean_len, token_bytes * hkv * total_pages * page,
                                                       rows, items, token_bytes, mfma))
        if resolved["balanced"] or resolved["pages_per_split"] is not None:
            # what a kernel without the balanced form falls back to
            split, chunk = decode_partition(batch, heads, hkv, max_pages, total_pages,
                                            quantized=k.dtype in _QUANT_DTYPES, q_len=q_len)
            resolved["split_k"] = split
            if resolved["pages_per_split"] is None:
                resolved["pages_per_split"] = chunk
            # A skewed batch cut into partitions of one size runs 4-wave
            # workgroups: the library's own choice (8 waves for partitions of
            # >= 1024 keys, measured on uniform batches) was 1.04-1.4x slower.
            if resolved["num_warps"] is None and is_ragged(batch, max_pages, total_pages):
                resolved["num_warps"] = 4
        else:
            resolved["split_k"], chosen = decode_split(items, max_len, mean_len, token_bytes, mfma, shared,
                                                       rows=rows, waves=waves)
            resolved["pages_per_split"] = 0
            if resolved["num_warps"] is None:
                resolved["num_warps"] = chosen
    if resolved["pages_per_split"] is None:
        resolved["pages_per_split"] = 0
    balanced = resolved["balanced"] = resolved["balanced"] or 0
    if not isinstance(balanced, int) or not 0 <= balanced <= 4096:
        raise ValueError(f"balanced must be an integer in [0, 4096], got {balanced}")
    split_k = resolved["split_k"]
    if not isinstance(split_k, int) or isinstance(split_k, bool) or split_k < 1:
        raise ValueError(f"split_k must be a positive integer, got {split_k}")
    if split_k > 64:
        raise ValueError(f"split_k must be <= 64, got {split_k}")
    pps = resolved["pages_per_split"]
    if not isinstance(pps, int) or isinstance(pps, bool) or pps < 0:
        raise ValueError(f"pages_per_split must be a non-negative integer, got {pps}")
    if resolved["num_warps"] not in (None, 1, 2, 4, 8, 16, 32):
        raise ValueError(f"num_warps must be a power of two <= 32, got {resolved['num_warps']}")
    if resolved["num_warps"] not in (None, 4, 8):
        raise ValueError(f"num_warps must be 4 or 8 waves per workgroup on MI355X, got {resolved['num_warps']}")
    if resolved["num_stages"] < 1:
        raise ValueError(f"num_stages must be >= 1, got {resolved['num_stages']}")
    if resolved["kernel"] not in _KERNEL_CODES:
        raise ValueError(f"kernel must be None, 'valu', 'mfma' or 'generic', got {resolved['kernel']!r}")
    if resolved["kernel"] in ("valu", "generic") and q_len > 1:
        raise ValueError(f"kernel {resolved['kernel']!r} takes one query per sequence; multi-token decode runs "
                         "on 'mfma'")
    if (resolved["kernel"] == "valu" and cache.k_cache.dtype in _QUANT_DTYPES
            and q.shape[-2] // cache.num_kv_heads >= 8):
        raise ValueError("kernel 'valu' takes int8/float8 caches only for GQA groups below 8; use 'mfma'")
    return resolved


def _validate_decode_inputs(q: torch.Tensor, cache: PagedKVCache, multi: bool = False,
                            prepare=None) -> tuple[int, int, tuple | None]:
    """``decode.py:503-522`` + ``paging.validate_cache``, with one host wait.

    ``multi``: ``q`` is ``[batch, q_len, heads, head_dim]`` and every sequence
    must already hold its q_len new tokens.  ``prepare``: called while the
    check kernel of ROCm tensors runs (its errors are left to the caller's
    own checks).  Returns ``(max_len, total_pages)`` for the partition
    heuristic and what ``prepare`` returned (None: not called, or it raised)."""
    if not isinstance(cache, PagedKVCache):
        raise TypeError("cache must be a PagedKVCache")
    _check_layout(cache)
    if multi:
        if q.dim() != 4:
            raise ValueError(f"q must be [batch, q_len, heads, head_dim], got {tuple(q.shape)}")
    elif q.dim() != 3:
        raise ValueError(f"q must be [batch, heads, head_dim], got {tuple(q.shape)}")
    if q.shape[0] != cache.batch_size:
        raise ValueError(f"q batch {q.shape[0]} != cache batch {cache.batch_size}")
    if q.shape[-1] != cache.head_dim:
        raise ValueError(f"q head_dim {q.shape[-1]} != cache head_dim {cache.head_dim}")
    if q.shape[-2] % cache.num_kv_heads != 0:
        raise ValueError(f"num_heads {q.shape[-2]} must be divisible by num_kv_heads {cache.num_kv_heads}")
    if q.device != cache.k_cache.device:
        raise ValueError("q and cache must live on the same device")
    if not q.is_floating_point():
        raise ValueError(f"q must be floating point, got {q.dtype}")
    sl, pt = cache.seq_lens, cache.page_table
    prepared = None
    if prepare is not None and sl.is_cuda and sl.is_contiguous() and pt.stride(-1) == 1 and pt.numel() \
            and _hip.is_loaded():
        check = _hip.check_begin(_hip.CHECK_CACHE, _hip.current_stream_handle(sl.device), sl.device, seq_lens=sl,
                                 page_table=pt, page_size=cache.page_size)
        try:
            prepared = prepare()
        except Exception:
            prepared = None
        r = check.wait()
        min_len, max_len, lo, hi, total_pages = r[0], r[1], r[12], r[13], r[2]
        if lo == _NO_PAGE:
            lo, hi = 0, -1
    else:
        min_len, max_len, lo, hi, total_pages = cache_stats(cache, with_total_pages=True)
    if min_len < 0:
        raise AssertionError("seq_lens must be non-negative")
    capacity = cache.capacity
    if max_len > capacity:
        raise AssertionError(f"seq_len {max_len} exceeds page-table capacity {capacity}")
    if max_len > 0:
        if lo < 0:
            raise AssertionError("page_table contains a negative page id")
        if hi >= cache.num_pages:
            raise AssertionError(f"page_table references page {hi} but cache has {cache.num_pages} pages")
    if min_len <= 0:
        raise ValueError("decode requires every sequence to hold at least one cached token")
    if multi and min_len < q.shape[1]:
        raise ValueError(f"multi-token decode requires every sequence to hold its {q.shape[1]} new tokens "
                         f"(shortest seq_len {min_len})")
    return max_len, total_pages, prepared


def _require_rocm(q: torch.Tensor, cache: PagedKVCache, what: str) -> None:
    tensors = (q, cache.k_cache, cache.v_cache, cache.page_table, cache.seq_lens)
    if not all(t.is_cuda for t in tensors):
        raise RuntimeError(
            f"{what}: inputs must be ROCm device tensors; this build runs the gfx950 HIP kernel only "
            "(no CPU or reference fallback)"
        )


# Split-K merge counters of the one-call decode paths: one zeroed int32
# buffer per (device, stream), grown on demand.  Every launch leaves its
# counters zero, so launches in one stream's order share them; launches on
# other streams get their own.
_MERGE_COUNTERS: dict[tuple[int, int], torch.Tensor] = {}


def merge_counters(q: torch.Tensor, split_k: int) -> torch.Tensor | None:
    """Zeroed merge counters for a split-K launch of ``q`` on torch's current
    stream (None when ``split_k`` is 1): the decode kernels then merge the
    partitions themselves instead of a second kernel."""
    if split_k <= 1:
        return None
    rows = q.shape[0] * (q.shape[1] if q.dim() == 4 else 1)
    n = rows * q.shape[-2]  # fat_paged_decode_counters_bytes / 4: one int32 per (query row, head)
    dev = q.device
    key = (dev.index if dev.index is not None else torch.cuda.current_device(), _hip.current_stream_handle(dev))
    t = _MERGE_COUNTERS.get(key)
    if t is None or t.numel() < n:
        t = torch.zeros(max(n, 4096), dtype=torch.int32, device=q.device)
        _MERGE_COUNTERS[key] = t
    return t


def paged_decode_launch(
    q: torch.Tensor,
    cache: PagedKVCache,
    softmax_scale: float,
    split_k: int,
    out: torch.Tensor | None = None,
    workspace: torch.Tensor | None = None,
    scales=None,
    waves_per_group: int | None = None,
    pages_per_split: int = 0,
    kernel: str | None = None,
    counters: torch.Tensor | None = None,
) -> torch.Tensor:
    """Enqueue the HIP decode without validation or synchronisation.

    ``q`` (``[B, H, D]``, or ``[B, T, H, D]`` for multi-token decode) must be
    contiguous fp16/bf16 on the cache's device; ``out`` (default
    ``empty_like(q)``) and ``workspace`` (default: allocated) may be passed in
    to avoid allocations.  ``kernel``: None (library's choice), ``"valu"`` or
    ``"mfma"``.  ``counters``: zeroed int32 split-K merge counters
    (:func:`merge_counters`, or any buffer of ``decode_counters_bytes`` that
    only this stream's launches use); the decode launch then merges its
    partitions itself.  None: a second kernel merges.
    """
    a, out, _keep = _decode_block(q, cache, softmax_scale, scales, out)
    _launch_block(a, q, split_k, workspace=workspace, waves_per_group=waves_per_group,
                  pages_per_split=pages_per_split, kernel=kernel, counters=counters)
    return out


def _decode_block(q, cache, softmax_scale, scales=None, out=None):
    """The argument block of a decode launch but for its partitions
    (:func:`_launch_block`), its output, and the tensors that have to live
    until the launch is enqueued."""
    if cache.k_cache.stride(-1) != 1 or cache.v_cache.stride(-1) != 1:
        raise ValueError("k_cache and v_cache need a contiguous head_dim axis")
    if out is None:
        out = torch.empty_like(q)
    # The kernels read page_table rows with a unit column stride and seq_lens
    # densely (the reference honours any strides, kernels/decode.py:89).
    pt = cache.page_table if cache.page_table.stride(-1) == 1 else cache.page_table.contiguous()
    sl = cache.seq_lens if cache.seq_lens.is_contiguous() else cache.seq_lens.contiguous()
    k_scale = v_scale = None
    if scales is not None:
        k_scale = scales["k"] if isinstance(scales, dict) else scales.k
        v_scale = scales["v"] if isinstance(scales, dict) else scales.v
    a = _hip.decode_args(q, cache.k_cache, cache.v_cache, pt, sl, out, cache.page_size, softmax_scale, 1,
                         k_scale=k_scale, v_scale=v_scale)
    return a, out, (q, pt, sl, k_scale, v_scale)


def _launch_block(a, q, split_k, workspace=None, waves_per_group=None, pages_per_split=0, kernel=None,
                  counters=None) -> None:
    """Enqueue the block of :func:`_decode_block` with these partitions."""
    rows = q.shape[0] * (q.shape[1] if q.dim() == 4 else 1)
    # fat_paged_decode_workspace_bytes: (acc, m, l) per (query row, head, partition)
    need = 4 * rows * q.shape[-2] * split_k * (q.shape[-1] + 2) if split_k > 1 else 0
    if need and (workspace is None or workspace.numel() * workspace.element_size() < need):
        workspace = torch.empty(need, dtype=torch.uint8, device=q.device)
    a.workspace = None if workspace is None else workspace.data_ptr()
    a.workspace_bytes = need  # held, as just checked
    # fat_paged_decode_counters_bytes: one int32 per (query row, head)
    if counters is not None and counters.numel() * counters.element_size() < 4 * rows * q.shape[-2]:
        raise ValueError("paged_decode_launch: counters smaller than decode_counters_bytes(rows, num_heads)")
    a.split_k = int(split_k)
    a.waves_per_group = waves_per_group or 0
    a.pages_per_split = int(pages_per_split)
    a.kernel = _KERNEL_CODES[kernel]
    a.merge_counters = None if counters is None else counters.data_ptr()
    _hip.decode_with_args(a, _hip.current_stream_handle(q.device))


def _balance(a, cfg) -> int:
    """Set up the block ``a`` for a balanced launch if ``cfg`` asks for one and
    the kernel has that form; returns its workspace bytes (0: it hasn't, and
    the block is for split_k partitions)."""
    if not cfg["balanced"]:
        return 0
    a.kernel = _KERNEL_CODES[cfg["kernel"]]
    a.balanced = cfg["balanced"]
    need = _hip.decode_balanced_workspace_bytes(a)
    if not need:
        a.balanced = 0
    return need


def _plan_workspace_bytes(a, cfg) -> int:
    """Set up the block ``a`` of a prepared launch as :func:`_balance` does and
    return the workspace bytes that cover each of its runs: a run whose query
    isn't 16-byte aligned can go to the generic kernel, which has no balanced
    form, and then takes ``a``'s partitions (0: neither form uses any)."""
    rows = a.batch * max(1, a.q_len)
    return max(_balance(a, cfg), _hip.decode_workspace_bytes(rows, a.num_heads, a.head_dim, cfg["split_k"]))


def _decode(q, cache, scale, cfg, prepared, scales=None) -> torch.Tensor:
    """Launch with the resolved partitions, from the prepared block if there
    is one."""
    if prepared is None:
        prepared = _decode_block(q.contiguous(), cache, scale, scales)
    a, out, keep = prepared
    q = keep[0]  # the copy that the block points at, where q wasn't contiguous
    need = _balance(a, cfg)
    if need:
        workspace = torch.empty(need, dtype=torch.uint8, device=q.device)
        a.workspace, a.workspace_bytes = workspace.data_ptr(), need
        a.merge_counters = merge_counters(q, 2).data_ptr()
        _hip.decode_with_args(a, _hip.current_stream_handle(q.device))
        del keep
        return out
    _launch_block(a, q, cfg["split_k"], waves_per_group=cfg["num_warps"], pages_per_split=cfg["pages_per_split"],
                  kernel=cfg["kernel"], counters=merge_counters(q, cfg["split_k"]))
    del keep
    return out


def _dense_scales(scales) -> dict:
    """``{"k", "v"}`` of QuantScales or such a dict, contiguous."""
    k_scale = scales["k"] if isinstance(scales, dict) else scales.k
    v_scale = scales["v"] if isinstance(scales, dict) else scales.v
    return {"k": k_scale.contiguous(), "v": v_scale.contiguous()}


def _scale_of(q, softmax_scale) -> float:
    return float(softmax_scale) if softmax_scale is not None else q.shape[-1] ** -0.5


def paged_decode_attention(
    q: torch.Tensor,
    cache: PagedKVCache,
    softmax_scale: float | None = None,
    config: dict | None = None,
    grouped: bool = False,
) -> torch.Tensor:
    """Paged decode attention, one query per sequence (``decode.py:533-642``).

    ``q``: ``[batch, num_heads, head_dim]`` fp16/bf16/fp32 on a ROCm device;
    the cache holds the same dtype (fp32 runs on the HIP kernel too, where the
    reference falls back to its fp32 oracle, ``decode.py:569-576``).  ``softmax_scale`` defaults to
    ``head_dim ** -0.5``.  ``config``: ``split_k`` (1 = no split; default from
    the MI355X heuristic), ``num_warps``, ``num_stages``.  ``grouped`` is
    accepted for compatibility: the HIP kernel always reads each K/V page
    once per GQA group.  Returns ``[batch, num_heads, head_dim]`` in
    ``q.dtype``.
    """
    del grouped  # every launch is grouped on MI355X
    max_len, total_pages, prepared = _validate_decode_inputs(
        q, cache, prepare=lambda: _decode_block(q.contiguous(), cache, _scale_of(q, softmax_scale)))
    scale = _scale_of(q, softmax_scale)
    cfg = _resolve_config(config, q, cache, max_len, total_pages)
    _require_rocm(q, cache, "paged_decode_attention")
    if q.dtype not in _DECODE_DTYPES:
        raise ValueError(f"paged_decode_attention: dtype {q.dtype} is not fp16/bf16/fp32 (the HIP kernels' types)")
    if cache.k_cache.dtype != q.dtype:
        raise ValueError(f"q dtype {q.dtype} must match cache dtype {cache.k_cache.dtype}")
    return _decode(q, cache, scale, cfg, prepared)


def paged_decode_attention_fp8(
    q: torch.Tensor,
    cache: PagedKVCache,
    scales,
    softmax_scale: float | None = None,
    config: dict | None = None,
) -> torch.Tensor:
    """Decode against an int8 / float8_e4m3fn cache (``decode.py:645-704``).

    ``scales`` is a :class:`~flashattntile_amd.quant.QuantScales` (or a dict
    with ``"k"``/``"v"``), fp32 ``[num_pages, num_kv_heads]``.  Pages are
    dequantised in registers as ``(float(x) * scale).to(q.dtype)``.
    """
    max_len, total_pages, prepared = _validate_decode_inputs(
        q, cache, prepare=lambda: _decode_block(q.contiguous(), cache, _scale_of(q, softmax_scale),
                                                _dense_scales(scales)))
    k_scale = scales["k"] if isinstance(scales, dict) else scales.k
    v_scale = scales["v"] if isinstance(scales, dict) else scales.v
    quant_dtype = cache.k_cache.dtype
    if quant_dtype not in _QUANT_DTYPES:
        raise ValueError(f"expected int8/float8 cache, got {quant_dtype}")
    expected = (cache.num_pages, cache.num_kv_heads)
    if tuple(k_scale.shape) != expected or tuple(v_scale.shape) != expected:
        raise ValueError(f"scales must have shape {expected}, got {tuple(k_scale.shape)}")
    scale = _scale_of(q, softmax_scale)
    cfg = _resolve_config(config, q, cache, max_len, total_pages)
    _require_rocm(q, cache, "paged_decode_attention_fp8")
    if not (k_scale.is_cuda and v_scale.is_cuda):
        raise RuntimeError("paged_decode_attention_fp8: scales must be ROCm device tensors")
    if q.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError(f"quantised decode requires fp16/bf16 queries, got {q.dtype}")
    if k_scale.dtype != torch.float32 or v_scale.dtype != torch.float32:
        raise ValueError("scales must be float32")
    return _decode(q, cache, scale, cfg, prepared, _dense_scales(scales) if prepared is None else None)


def paged_decode_attention_multi(
    q: torch.Tensor,
    cache: PagedKVCache,
    softmax_scale: float | None = None,
    config: dict | None = None,
    scales=None,
) -> torch.Tensor:
    """Multi-token (speculative) decode: ``q`` ``[batch, q_len, num_heads,
    head_dim]`` holds the last q_len tokens of each sequence, whose K/V are
    already in ``cache`` (``seq_lens[b] >= q_len``).  Token t of sequence b
    attends keys ``j <= seq_lens[b] - q_len + t`` -- the bottom-right causal
    convention of :func:`~flashattntile_amd.kernels.prefill.prefill_attention`
    -- and every K/V page is read once per KV head (per 32 (head, token)
    rows) by the MFMA decode kernel.  ``scales`` (QuantScales or
    ``{"k", "v"}``) selects an int8/float8_e4m3fn cache.  ``config`` as for
    :func:`paged_decode_attention`.  Returns ``q``'s shape and dtype.
    """
    max_len, total_pages, prepared = _validate_decode_inputs(
        q, cache, multi=True, prepare=lambda: _decode_block(q.contiguous(), cache, _scale_of(q, softmax_scale),
                                                            None if scales is None else _dense_scales(scales)))
    q_len = int(q.shape[1])
    if q_len > 64:
        raise ValueError(f"multi-token decode takes at most 64 tokens per sequence, got {q_len}")
    quantized = cache.k_cache.dtype in _QUANT_DTYPES
    if quantized != (scales is not None):
        raise ValueError("an int8/float8 cache needs scales, and only such a cache takes them")
    scale = _scale_of(q, softmax_scale)
    cfg = _resolve_config(config, q, cache, max_len, total_pages, q_len=q_len)
    _require_rocm(q, cache, "paged_decode_attention_multi")
    if q.dtype not in (torch.float16, torch.bfloat16):
        raise ValueError(f"paged_decode_attention_multi: dtype {q.dtype} is not fp16/bf16")
    sc = None
    if quantized:
        k_scale = scales["k"] if isinstance(scales, dict) else scales.k
        v_scale = scales["v"] if isinstance(scales, dict) else scales.v
        expected = (cache.num_pages, cache.num_kv_heads)
        if tuple(k_scale.shape) != expected or tuple(v_scale.shape) != expected:
            raise ValueError(f"scales must have shape {expected}, got {tuple(k_scale.shape)}")
        if k_scale.dtype != torch.float32 or v_scale.dtype != torch.float32:
            raise ValueError("scales must be float32")
        sc = _dense_scales(scales) if prepared is None else None
    elif cache.k_cache.dtype != q.dtype:
        raise ValueError(f"q dtype {q.dtype} must match cache dtype {cache.k_cache.dtype}")
    return _decode(q, cache, scale, cfg, prepared, sc)


# Streams, other than the one a plan was made on, whose workspace it keeps;
# captures that find cleared counters ready.
_MAX_STREAMS = 64
_CAPTURE_COUNTERS = 4


def _on_stream(stream: int, device: torch.device):
    """Make the stream with this handle torch's current one."""
    if stream == _hip.current_stream_handle(device):
        return contextlib.nullcontext()
    return torch.cuda.stream(torch.cuda.ExternalStream(stream, device=device) if stream
                             else torch.cuda.default_stream(device))


class _StreamState:
    """What the runs of a :class:`DecodeLaunch` on one stream, or in one
    capture of it, use: their argument block, workspace and merge counters
    (both None where the launch has no partitions to merge)."""

    __slots__ = ("args", "workspace", "counters")

    def __init__(self, args, workspace, counters) -> None:
        self.args = type(args).from_buffer_copy(args)
        _hip.set_workspace(self.args, workspace)
        self.args.merge_counters = None if counters is None else counters.data_ptr()
        self.workspace, self.counters = workspace, counters


class DecodeLaunch:
    """A decode launch prepared once and run every step (plan / run).

    Construction validates ``q`` and ``cache`` (one synchronisation, as
    :func:`paged_decode_attention` does, unless ``max_len`` and
    ``total_pages`` are given), resolves the launch (``config``, else the
    tuned store, else the heuristic), allocates the workspace and fills the
    ``fat_decode_args`` block.  :meth:`run` then only writes the
    query and output addresses into that block and enqueues
    ``fat_paged_decode``: no validation, synchronisation or allocation, about
    the cost of one ctypes call.

    Runs on different streams, captured runs among them, may overlap: each
    stream but the one that was current at construction, and each capture,
    gets a workspace and merge counters of its own at its first run (the plan
    keeps those of the last 64 streams, and a capture's as long as it lives:
    it has to outlive its graphs, as the cache has).  Runs on one stream share
    theirs; no two threads may run a plan on one stream at a time.

    The page table and seq_lens are read on the
    device at every run, so the serving engine updates them in place.  ``q``
    and ``out`` passed to :meth:`run` must have the dtype, shape and strides
    of the ``q`` given here (``out``: contiguous).  ``q`` is ``[B, H, D]`` or
    ``[B, T, H, D]`` (multi-token decode); ``scales`` selects an int8 /
    float8_e4m3fn cache.
    """

    def __init__(self, q: torch.Tensor, cache: PagedKVCache, softmax_scale: float | None = None,
                 config: dict | None = None, scales=None, max_len: int | None = None,
                 total_pages: int | None = None) -> None:
        multi = q.dim() == 4
        if max_len is None or total_pages is None:
            max_len, total_pages, _ = _validate_decode_inputs(q, cache, multi=multi)
        q_len = int(q.shape[1]) if multi else 1
        cfg = _resolve_config(config, q, cache, max_len, total_pages, q_len=q_len)
        _require_rocm(q, cache, "DecodeLaunch")
        quantized = cache.k_cache.dtype in _QUANT_DTYPES
        if q.dtype not in (_DECODE_DTYPES[:2] if quantized else _DECODE_DTYPES):
            raise ValueError(f"DecodeLaunch: q dtype {q.dtype} is not one the HIP decode takes for a "
                             f"{cache.k_cache.dtype} cache")
        if quantized != (scales is not None):
            raise ValueError("an int8/float8 cache needs scales, and only such a cache takes them")
        if not quantized and cache.k_cache.dtype != q.dtype:
            raise ValueError(f"q dtype {q.dtype} must match cache dtype {cache.k_cache.dtype}")
        if not q.is_contiguous():
            raise ValueError("DecodeLaunch: q must be contiguous")
        k_scale = v_scale = None
        if quantized:
            k_scale = (scales["k"] if isinstance(scales, dict) else scales.k).contiguous()
            v_scale = (scales["v"] if isinstance(scales, dict) else scales.v).contiguous()
            expected = (cache.num_pages, cache.num_kv_heads)
            if tuple(k_scale.shape) != expected or tuple(v_scale.shape) != expected:
                raise ValueError(f"scales must have shape {expected}, got {tuple(k_scale.shape)}")
            if k_scale.dtype != torch.float32 or v_scale.dtype != torch.float32:
                raise ValueError("scales must be float32")
        if cache.k_cache.stride(-1) != 1 or cache.v_cache.stride(-1) != 1:
            raise ValueError("k_cache and v_cache need a contiguous head_dim axis")
        # The argument block points at the engine's own table and lengths,
        # which it updates in place: they cannot be copied to a dense layout.
        if cache.page_table.stride(-1) != 1 or not cache.seq_lens.is_contiguous():
            raise ValueError("DecodeLaunch: page_table rows and seq_lens must be contiguous")
        self.config = cfg
        self.softmax_scale = float(softmax_scale) if softmax_scale is not None else q.shape[-1] ** -0.5
        self._args = _hip.decode_args(q, cache.k_cache, cache.v_cache, cache.page_table, cache.seq_lens, q,
                                      cache.page_size, self.softmax_scale, cfg["split_k"], k_scale=k_scale,
                                      v_scale=v_scale, waves_per_group=cfg["num_warps"] or 0,
                                      pages_per_split=cfg["pages_per_split"], kernel=_KERNEL_CODES[cfg["kernel"]])
        self._need = _plan_workspace_bytes(self._args, cfg)
        self._num_counters = _hip.decode_counters_bytes(q.shape[0] * q_len, q.shape[-2]) // 4
        self._keep = (cache, k_scale, v_scale)  # the argument block points into these
        self._shape, self._dtype = tuple(q.shape), q.dtype
        self._device = q.device
        self._lock = threading.Lock()
        self._states: dict[tuple[int, int], _StreamState] = {}
        self._cleared: torch.Tensor | None = None
        self._cleared_sets = 0
        stream = _hip.current_stream_handle(q.device)
        self._home = (stream, _hip.stream_capture_id(stream) if self._need else 0)
        if self._need and not self._home[1]:
            # For this stream, and for captures, which then need no fill of
            # their own (a launch more in every replay).
            self._cleared_sets = 1 + _CAPTURE_COUNTERS
            self._cleared = self._zero_counters(self._cleared_sets)
        home = self._add_state(self._home)
        self.workspace, self.counters = home.workspace, home.counters

    def _zero_counters(self, sets: int) -> torch.Tensor:
        return torch.zeros(sets, self._num_counters, dtype=torch.int32, device=self._device)

    def _state(self, stream: int) -> _StreamState:
        key = (stream, _hip.stream_capture_id(stream) if self._need else 0)
        return self._states.get(key) or self._add_state(key)

    def _add_state(self, key: tuple[int, int]) -> _StreamState:
        stream, capture = key
        with self._lock:
            state = self._states.get(key)
            if state is not None:
                return state
            workspace = counters = None
            if self._need:
                # Allocated and cleared on the stream that uses them: their
                # memory goes to another use only behind its last run there.
                with _on_stream(stream, self._device):
                    workspace = torch.empty(self._need, dtype=torch.uint8, device=self._device)
                    if self._cleared_sets and (capture or key == self._home):
                        self._cleared_sets -= 1
                        counters = self._cleared[self._cleared_sets]
                    else:
                        counters = self._zero_counters(1)[0]
            if not capture and len(self._states) > _MAX_STREAMS:
                eager = [k for k in self._states if not k[1] and k != self._home]
                if len(eager) >= _MAX_STREAMS:
                    del self._states[eager[0]]
            state = self._states[key] = _StreamState(self._args, workspace, counters)
            return state

    def run(self, q: torch.Tensor, out: torch.Tensor | None = None, stream: int | None = None) -> torch.Tensor:
        """Decode ``q`` into ``out`` (default: a new tensor) on ``stream``
        (a hipStream_t handle; default torch's current stream)."""
        if tuple(q.shape) != self._shape or q.dtype != self._dtype or not q.is_contiguous():
            raise ValueError(f"DecodeLaunch.run: q must be a contiguous {self._dtype} tensor of shape {self._shape}")
        if out is None:
            out = torch.empty_like(q)
        elif tuple(out.shape) != self._shape or out.dtype != self._dtype or not out.is_contiguous():
            raise ValueError(f"DecodeLaunch.run: out must be a contiguous {self._dtype} tensor of shape {self._shape}")
        if stream is None:
            stream = _hip.current_stream_handle(self._device)
        state = self._state(stream)
        a = state.args
        a.q = q.data_ptr()
        a.out = out.data_ptr()
        _hip.decode_with_args(a, stream)
        return out
