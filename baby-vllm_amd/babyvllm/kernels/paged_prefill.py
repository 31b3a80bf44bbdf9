"""Varlen paged prefill attention on the HIP kernel (drop-in for babyvllm/kernels/paged_prefill.py:104-146).

``paged_prefill_attention(q, kv_cache, md, scale)`` keeps the reference's
signature and semantics: a flattened batch of sequences, each with
``context_lens[s]`` cached tokens plus ``q_len`` new query rows, causal, GQA,
with K/V (prefix and new tokens alike) read from the paged cache through
``md.block_tables``. Decode rows (query length 1) may be mixed into the step.

Few new tokens behind long prefixes run in key ranges, and long uneven decode rows
in chunks, chosen from the step's host lists and the live lengths: the bits of such
a sequence depend on the other sequences of the step, within the rounding of fp32
sums in another order. Both take fp32 scratch (key ranges at most 64 MiB); without
the memory for it the launch that needs none runs.
"""

from __future__ import annotations

import torch

from babyvllm.kernels import _lib


def _single_query_seqs(md, num_seqs):
    """Sequences with exactly one query token, from the host copy of query_start_loc.

    -1 (unknown) when the metadata carries no host copy of the right length;
    the library then checks every sequence on the device.
    """
    qsl = getattr(md, "query_start_loc_cpu", None)
    if qsl is None or len(qsl) != num_seqs + 1:
        return -1
    return sum(1 for i in range(num_seqs) if qsl[i + 1] - qsl[i] == 1)


# Narrower tables never split: their sequences are a few key tiles long.
_SPLIT_MIN_PAGES = 32


def _key_tiles(md, num_seqs, num_heads, num_kv_heads):
    """(64-key tiles that the blocks of the sequences of several queries cover, tiles of the
    longest of them) from the host lists, -1 for each if those are absent or of another length."""
    qsl, seq = getattr(md, "query_start_loc_cpu", None), getattr(md, "seq_lens_cpu", None)
    if qsl is None or seq is None or len(seq) != num_seqs or len(qsl) != num_seqs + 1:
        return -1, -1
    group, tiles, longest = num_heads // num_kv_heads, 0, 0
    for i in range(num_seqs):
        n = qsl[i + 1] - qsl[i]
        if n > 1:
            keys = (int(seq[i]) + 63) >> 6
            tiles += ((int(n) * group + 127) >> 7) * keys
            longest = max(longest, keys)
    return tiles, longest


def _split_tiles(md, num_seqs, num_tokens, single, num_heads, num_kv_heads, head_dim, width):
    """Key tiles per range of a split launch, 0 for the plain one.

    The choice looks at the work the host lists describe (the table's width stands in
    for lists that are absent or of another length); the results do not depend on them.
    """
    if width < _SPLIT_MIN_PAGES:
        return 0
    tiles, longest = _key_tiles(md, num_seqs, num_heads, num_kv_heads)
    return _lib.lib().bvllm_prefill_split_tiles(num_seqs, num_tokens, int(md.max_query_len), single, num_heads,
                                                num_kv_heads, head_dim, width, tiles, longest)


def _balance_rows(md, num_seqs, num_heads, num_kv_heads, split_tiles=0):
    """Whether the single-query rows are cut into chunks (also a choice by the host lists);
    ``split_tiles`` is the key range that the other sequences are cut into, 0 if they are whole."""
    qsl, seq = getattr(md, "query_start_loc_cpu", None), getattr(md, "seq_lens_cpu", None)
    if qsl is None or seq is None or len(seq) != num_seqs or len(qsl) != num_seqs + 1:
        return 0
    pages = [(int(seq[i]) + 15) // 16 for i in range(num_seqs) if qsl[i + 1] - qsl[i] == 1]
    if not pages:
        return 0
    tiles = _key_tiles(md, num_seqs, num_heads, num_kv_heads)[1]
    if split_tiles > 0:
        tiles = min(split_tiles, tiles)
    return _lib.lib().bvllm_prefill_balance_rows(num_heads, num_kv_heads, max(pages), sum(pages), tiles)


def paged_prefill_attention(q, kv_cache, md, scale):
    """Causal attention for a flattened varlen batch, reading K/V from the paged cache.

    K/V of the step's tokens must already be in the cache (the RoPE + append
    kernel writes them first).
    """
    if q.is_cuda:
        out = _lib.fast().prefill(q, kv_cache, md.block_tables, md.query_start_loc, md.seq_lens, md.context_lens,
                                  getattr(md, "query_start_loc_cpu", None), getattr(md, "seq_lens_cpu", None),
                                  md.max_query_len, scale, _SPLIT_MIN_PAGES, *_lib.current())
        if out is not None:
            return out
    num_tokens, num_heads, head_dim = q.shape
    num_kv_heads = kv_cache.shape[3]
    page = kv_cache.shape[2]
    assert head_dim & (head_dim - 1) == 0, f"head_dim {head_dim} must be a power of two"
    assert num_heads % num_kv_heads == 0

    for name, t in (("q", q), ("kv_cache", kv_cache), ("block_tables", md.block_tables),
                    ("query_start_loc", md.query_start_loc), ("seq_lens", md.seq_lens),
                    ("context_lens", md.context_lens)):
        _lib.require_rocm_tensor(name, t)
    if q.dtype != torch.bfloat16 or kv_cache.dtype != torch.bfloat16:
        raise TypeError("q and kv_cache must be bfloat16")
    if q.stride(-1) != 1:
        raise ValueError("q must have a unit last stride")
    for name, t in (("block_tables", md.block_tables), ("query_start_loc", md.query_start_loc),
                    ("seq_lens", md.seq_lens), ("context_lens", md.context_lens)):
        if t.dtype != torch.int32:
            raise TypeError(f"{name} must be int32, got {t.dtype}")
    bt = md.block_tables
    if bt.dim() != 2 or bt.stride(1) != 1:
        raise ValueError("block_tables must be [S, W] with a unit last stride")
    qsl = md.query_start_loc.contiguous()
    seq_lens = md.seq_lens.contiguous()
    ctx_lens = md.context_lens.contiguous()

    out = torch.empty(num_tokens, num_heads, head_dim, device=q.device, dtype=q.dtype)
    if num_tokens == 0:
        return out
    k_cache, v_cache = kv_cache[0], kv_cache[1]
    if k_cache.stride() != v_cache.stride() or k_cache.stride(3) != 1:
        raise ValueError("K and V halves of kv_cache must share a layout with unit last stride")
    num_seqs = seq_lens.shape[0]
    single = _single_query_seqs(md, num_seqs)
    split_tiles = _split_tiles(md, num_seqs, num_tokens, single, num_heads, num_kv_heads, head_dim, bt.shape[1])
    args = (
        q.data_ptr(), q.stride(0), q.stride(1),
        k_cache.data_ptr(), v_cache.data_ptr(), k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
        kv_cache.shape[1],
        bt.data_ptr(), bt.stride(0), bt.shape[1],
        qsl.data_ptr(), seq_lens.data_ptr(), ctx_lens.data_ptr(), float(scale),
        out.data_ptr(), out.stride(0), out.stride(1),
        num_seqs, num_tokens, int(md.max_query_len), single,
        num_heads, num_kv_heads, head_dim, page,
    )
    h = _lib.lib()
    balance = 0
    if single > 0 and num_seqs * bt.shape[1] <= _lib.BALANCED_MAX_PAGES:
        balance = _balance_rows(md, num_seqs, num_heads, num_kv_heads, split_tiles)
    workspace = None
    if split_tiles > 0 or balance:
        ranges = 0
        if split_tiles > 0:
            longest = _key_tiles(md, num_seqs, num_heads, num_kv_heads)[1]
            ranges = h.bvllm_prefill_ranges(bt.shape[1], split_tiles, longest)
        nbytes = h.bvllm_prefill_workspace_bytes(num_seqs, num_tokens, num_heads, num_kv_heads, head_dim, ranges,
                                                 balance)
        workspace = _lib.optional_scratch(nbytes, q.device)
    if workspace is not None:
        rc = h.bvllm_paged_prefill_split(*args, workspace.data_ptr(), split_tiles, ranges, balance,
                                         _lib.stream_handle(q.device))
    else:
        rc = h.bvllm_paged_prefill(*args, _lib.stream_handle(q.device))
    _lib.check(rc, "bvllm_paged_prefill")
    return out
