"""Causal chunk / varlen prefill over a paged FP8 E4M3 KV cache (drop-in for
``microserve/layers/fp8_chunk_prefill_attention.py``), backed by the gfx950
FP8-MFMA HIP kernel."""

from __future__ import annotations

import torch

from microserve_amd import _lib


def _check_common(query, k_cache, v_cache, k_scale_cache, v_scale_cache):
    _, num_q_heads, head_dim = query.shape
    num_kv_heads = k_cache.shape[2]
    assert query.dtype in (torch.float16, torch.bfloat16)
    assert k_cache.dtype == v_cache.dtype == torch.float8_e4m3fn
    assert k_scale_cache.dtype == v_scale_cache.dtype == torch.float32
    assert num_q_heads % num_kv_heads == 0
    assert head_dim == k_cache.shape[3]
    for t in (k_cache, v_cache, k_scale_cache, v_scale_cache):
        assert t.is_contiguous(), "caches must be contiguous"
    _lib.on_device("prefill attention", query, k_cache, v_cache, k_scale_cache,
                   v_scale_cache)


def _launch(lib, what, query, caches, tables, cu_q, cu_k, prefix_len, output, num_seqs,
            max_seqlen_q, max_seqlen_k, max_blocks, softmax_scale):
    """One prefill launch.  The split partials' workspace, where the shapes
    need one, is allocated per call on the current stream, which the kernels
    run on: the caching allocator reuses it in stream order, and a graph
    capture takes it from its own pool."""
    k_cache, v_cache, k_scale_cache, v_scale_cache = caches
    total_q, num_q_heads, head_dim = query.shape
    num_blocks, block_size, num_kv_heads = k_cache.shape[:3]
    ws_bytes = lib.mskv_fp8_prefill_bounded_workspace_bytes(
        num_seqs, total_q, max_seqlen_q, max_seqlen_k, num_q_heads, num_kv_heads, head_dim,
        block_size, max_blocks)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=query.device) if ws_bytes else None
    status = lib.mskv_fp8_prefill_attention_bounded(
        query.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
        k_scale_cache.data_ptr(), v_scale_cache.data_ptr(), tables.data_ptr(),
        None if cu_q is None else cu_q.data_ptr(), None if cu_k is None else cu_k.data_ptr(),
        prefix_len, output.data_ptr(), num_seqs, total_q, max_seqlen_q, max_seqlen_k,
        num_q_heads, num_kv_heads, head_dim, block_size, num_blocks, max_blocks,
        float(softmax_scale),
        _lib.act_dtype(query), None if ws is None else ws.data_ptr(), ws_bytes,
        _lib.stream_of(query))
    _lib.check(status, what)


def fp8_chunk_prefill_attention(
    query: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
    k_scale_cache: torch.Tensor, v_scale_cache: torch.Tensor,
    block_table: torch.Tensor, prefix_len: int, softmax_scale: float,
    block_m: int | None = None, block_n: int | None = None,
) -> torch.Tensor:
    """Single-sequence causal chunk prefill, the reference's signature.

    ``query`` ``[Lq, H_q, D]`` attends over ``prefix_len + Lq`` cached
    positions read through the flattened ``block_table``
    (``fp8_chunk_prefill_attention.py:70-109``); query ``i`` sees positions
    ``< prefix_len + i + 1``.  ``block_m``/``block_n`` are accepted and
    ignored.  QK^T runs as FP8 MFMA contractions (the query split into exact
    e4m3 parts, the K bytes as stored); PV runs on the fp16 MFMA, with V's
    bytes converted to fp16 exactly and fp16 probability weights, which at
    the same matrix-core time as two FP8 parts of P keeps 11 significant
    bits for every weight.
    """
    del block_m, block_n
    res = _lib.fast.prefill(query, k_cache, v_cache, k_scale_cache, v_scale_cache, block_table,
                              None, None, prefix_len, 0, 0, softmax_scale)
    if res is not None:
        return res
    query = _lib.aligned(query)
    block_table = block_table.contiguous().view(-1)
    query_len = query.shape[0]
    _check_common(query, k_cache, v_cache, k_scale_cache, v_scale_cache)
    assert block_table.dtype == torch.int32
    _lib.on_device("fp8_chunk_prefill_attention", query, block_table)
    prefix_len = int(prefix_len)
    assert prefix_len >= 0
    output = torch.empty_like(query)
    if query_len == 0:
        return output
    _launch(_lib.load(), "fp8_chunk_prefill_attention", query,
            (k_cache, v_cache, k_scale_cache, v_scale_cache), block_table, None, None, prefix_len,
            output, 1, query_len, prefix_len + query_len, block_table.numel(),
            softmax_scale)
    return output


def fp8_varlen_prefill_attention(
    query: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
    k_scale_cache: torch.Tensor, v_scale_cache: torch.Tensor,
    block_tables: torch.Tensor, cu_seqlens_q: torch.Tensor,
    cu_seqlens_k: torch.Tensor, max_seqlen_q: int, softmax_scale: float,
    max_seqlen_k: int | None = None,
) -> torch.Tensor:
    """Varlen causal prefill with cached prefixes, in one launch.

    The batch the runner describes with ``cu_seqlens_q``/``cu_seqlens_k``
    (``model_runner.py:184-192``): sequence ``s`` owns query rows
    ``cu_seqlens_q[s]:cu_seqlens_q[s+1]`` and ``Lk = cu_seqlens_k[s+1] -
    cu_seqlens_k[s]`` cached positions (its new tokens included, since they
    are stored first); query ``i`` sees positions ``< Lk - Lq + i + 1``.
    ``block_tables`` is int32 ``[num_seqs, max_blocks]``.  ``max_seqlen_q``
    is a host integer, as in the reference's ``Context``.  ``max_seqlen_k``,
    the most cached positions of any sequence, only chooses how many ranges
    small batches split the keys into; without it the tables' width stands
    in, which costs short sequences under much wider tables a few
    microseconds (16 x 8 new over 100 cached tokens: 11.9 against 8.8).
    """
    bound = 0 if max_seqlen_k is None else int(max_seqlen_k)
    res = _lib.fast.prefill(query, k_cache, v_cache, k_scale_cache, v_scale_cache, block_tables,
                              cu_seqlens_q, cu_seqlens_k, 0, max_seqlen_q, bound,
                              softmax_scale)
    if res is not None:
        return res
    query = _lib.aligned(query)
    block_tables = block_tables.contiguous()
    cu_seqlens_q = cu_seqlens_q.contiguous()
    cu_seqlens_k = cu_seqlens_k.contiguous()
    total_q = query.shape[0]
    _check_common(query, k_cache, v_cache, k_scale_cache, v_scale_cache)
    assert block_tables.dtype == cu_seqlens_q.dtype == cu_seqlens_k.dtype == torch.int32
    num_seqs = cu_seqlens_q.numel() - 1
    assert cu_seqlens_k.numel() == num_seqs + 1
    assert block_tables.dim() == 2 and block_tables.shape[0] == num_seqs
    _lib.on_device("fp8_varlen_prefill_attention", query, block_tables, cu_seqlens_q,
                   cu_seqlens_k)
    output = torch.empty_like(query)
    if total_q == 0 or num_seqs == 0:
        return output
    _launch(_lib.load(), "fp8_varlen_prefill_attention", query,
            (k_cache, v_cache, k_scale_cache, v_scale_cache), block_tables, cu_seqlens_q,
            cu_seqlens_k, 0, output, num_seqs, int(max_seqlen_q), max(bound, 0),
            block_tables.shape[1], softmax_scale)
    return output
