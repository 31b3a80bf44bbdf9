"""Paged decode attention on the HIP kernel (drop-in for babyvllm/kernels/paged_attn.py:254-346).

``paged_decode_attention(q, kv_cache, block_tables, seq_lens, scale,
max_seq_len=None, partition_blocks=None)`` keeps the reference's signature:
one query token per sequence, GQA, pages read through the block table, and
the flash-decoding split chosen by ``decode_split_plan`` from the context
*bucket* (``max_seq_len``) and the batch's power-of-two bucket, never from the
live lengths, so the launch is identical on every replay of a captured graph.
Within it, a plan of one split with a bucket above ``BALANCE_MIN_PAGES`` and at most two
walks per CU (``balance_pays``) lets the device cut rows of more than 128 pages into chunks by the live lengths of the whole
batch: such a row's bits depend on the other rows' lengths too. ``partition_blocks=0``
(or the environment's "0") keeps one work-group per row and KV head, whose bits
depend on the row alone.

The wrapper allocates the output and, for a split launch, the fp32 partial
scratch through torch (so both land in a graph's private pool under capture),
then makes one C-ABI call on the current stream: no host synchronisation and
no device-to-host read.
"""

from __future__ import annotations

import functools
import os

import torch

from babyvllm.kernels import _lib
from babyvllm.kernels.decode_split import DECODE_PARTITION_ENV, MIN_PARTITION_BLOCKS, decode_split_plan, pow2_at_least

# A single-pass plan ("auto") sized for more pages than this runs the balanced launch
# (bvllm_paged_decode_balanced). Shorter rows can lose less to each other than its second
# launch costs equal ones (64 x 2048: 45.1 against 46.4 us; 64 rows of 200 to 2048: 30.2
# against 27.1; 64 of 100 to 4096: 52 against 34; 64 x 4096: 86.7 against 87.7).
BALANCE_MIN_PAGES = 128


def balance_pays(batch: int, n_heads: int, n_kv_heads: int, num_sms: int) -> bool:
    """At most two walks of a (row, 16 query heads of a KV head) per CU, so that one can be
    left alone on the card. With more, the plain launch evens the rows out by itself: over
    random batches of up to two per CU the balanced one takes 0.54 to 0.91 of its time on
    ragged rows, beyond 2.5 it is 2% slower on average and never pays (160 rows, 4 KV heads).
    The batch counts as the next power of two, as in the plan, so that an eager step and its
    graph agree."""
    if n_kv_heads < 1 or n_heads % n_kv_heads:
        return False
    return pow2_at_least(batch) * n_kv_heads * -(-n_heads // n_kv_heads // 16) <= 2 * num_sms


@functools.lru_cache(maxsize=None)
def _num_sms(device_index: int) -> int:
    return torch.cuda.get_device_properties(device_index).multi_processor_count


def _device_index(t: torch.Tensor) -> int:
    return t.device.index if t.device.index is not None else torch.cuda.current_device()


def paged_decode_attention(q, kv_cache, block_tables, seq_lens, scale,
                           max_seq_len=None, partition_blocks=None):
    """``[B, H, D]`` attention of one query token per row against its paged K/V.

    ``max_seq_len`` is the context bucket the step was sized for; it sets the
    split count. ``partition_blocks`` overrides BABYVLLM_DECODE_PARTITION.
    Rows with ``seq_len == 0`` return zeros.
    """
    if partition_blocks is None and q.is_cuda:
        d, stream = _lib.current()
        out = _lib.fast().decode(q, kv_cache, block_tables, seq_lens, scale, max_seq_len, _num_sms(d),
                                 MIN_PARTITION_BLOCKS, BALANCE_MIN_PAGES, DECODE_PARTITION_ENV, d, stream)
        if out is not None:
            return out
    for name, t in (("q", q), ("kv_cache", kv_cache), ("block_tables", block_tables),
                    ("seq_lens", seq_lens)):
        _lib.require_rocm_tensor(name, t)
    if q.dim() != 3 or q.stride(-1) != 1:
        raise ValueError("q must be [B, H, D] with a unit last stride")
    if q.dtype != torch.bfloat16 or kv_cache.dtype != torch.bfloat16:
        raise TypeError("q and kv_cache must be bfloat16")
    if block_tables.dtype != torch.int32 or seq_lens.dtype != torch.int32:
        raise TypeError("block_tables and seq_lens must be int32")
    if kv_cache.dim() != 5 or kv_cache.shape[0] != 2:
        raise ValueError(f"kv_cache must be [2, NB, BS, Hkv, D], got {tuple(kv_cache.shape)}")
    B, n_heads, head_dim = q.shape
    _, num_blocks, block_size, n_kv_heads, cache_dim = kv_cache.shape
    if cache_dim != head_dim:
        raise ValueError("kv_cache head_dim differs from q")
    if block_tables.dim() != 2 or block_tables.shape[0] < B or block_tables.stride(1) != 1:
        raise ValueError("block_tables must be [B, W] with a unit last stride")
    if seq_lens.dim() != 1 or seq_lens.shape[0] < B or not seq_lens.is_contiguous():
        raise ValueError("seq_lens must be a contiguous [B] vector")
    k_cache, v_cache = kv_cache[0], kv_cache[1]
    if k_cache.stride() != v_cache.stride() or k_cache.stride(3) != 1:
        raise ValueError("K and V halves of kv_cache must share a layout with unit last stride")

    width = block_tables.shape[1]
    num_splits, blocks_per_split = decode_split_plan(
        B, n_kv_heads, block_size, width, max_seq_len, _num_sms(_device_index(q)), partition_blocks,
    )
    out = torch.empty(B, n_heads, head_dim, device=q.device, dtype=q.dtype)
    if B == 0:
        return out
    h = _lib.lib()
    args = (
        q.data_ptr(), q.stride(0), q.stride(1),
        k_cache.data_ptr(), v_cache.data_ptr(), k_cache.stride(0), k_cache.stride(1), k_cache.stride(2),
        num_blocks,
        block_tables.data_ptr(), block_tables.stride(0), width,
        seq_lens.data_ptr(), float(scale),
        out.data_ptr(), out.stride(0), out.stride(1),
    )
    balanced = num_splits == 1 and blocks_per_split > BALANCE_MIN_PAGES and partition_blocks is None \
        and balance_pays(B, n_heads, n_kv_heads, _num_sms(_device_index(q))) \
        and B * width <= _lib.BALANCED_MAX_PAGES and os.environ.get(DECODE_PARTITION_ENV, "auto") == "auto"
    workspace = None
    if balanced:
        nbytes = h.bvllm_decode_balanced_workspace_bytes(B, n_heads, n_kv_heads, head_dim)
        workspace = _lib.optional_scratch(nbytes, q.device) if nbytes > 0 else None
        balanced = workspace is not None
    if not balanced:
        nbytes = h.bvllm_decode_workspace_bytes(B, n_heads, n_kv_heads, head_dim, num_splits, blocks_per_split)
        workspace = torch.empty(nbytes // 4, device=q.device, dtype=torch.float32) if nbytes > 0 else None
    ws = None if workspace is None else workspace.data_ptr()
    stream = _lib.stream_handle(q.device)
    if balanced:
        rc = h.bvllm_paged_decode_balanced(*args, ws, B, n_heads, n_kv_heads, head_dim, block_size, stream)
    else:
        rc = h.bvllm_paged_decode(*args, ws, num_splits, blocks_per_split,
                                  B, n_heads, n_kv_heads, head_dim, block_size, 0, stream)
    _lib.check(rc, "bvllm_paged_decode")
    return out
