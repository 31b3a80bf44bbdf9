"""A model's input rows on the HIP kernel (embed_tokens and rotary_emb of babyvllm/models/qwen2.py:109-118).

``embed_rows(ids, table, positions, cos_table, sin_table)`` returns ``(table[ids],
cos_table[positions], sin_table[positions])`` in bf16 from one launch, or ``None`` when
the call is not one for the kernel (the caller then takes torch's own operations): it
takes plain contiguous tensors on the current ROCm device, a bf16 embedding table and
fp32 cos/sin tables, outside autograd and every mode that has to see torch operations.
"""

from __future__ import annotations

import torch

from babyvllm.kernels import _lib
from babyvllm.kernels.linear import torch_must_see


def embed_rows(ids, table, positions, cos_table, sin_table):
    tensors = (ids, table, positions, cos_table, sin_table)
    if not ids.is_cuda or torch_must_see(*tensors):
        return None
    d, stream = _lib.current()
    for t, dtype, dim in zip(tensors, (torch.int64, torch.bfloat16, torch.int64, torch.float32, torch.float32),
                             (1, 2, 1, 2, 2)):
        if type(t) not in (torch.Tensor, torch.nn.Parameter) or not t.is_cuda or t.device.index != d \
                or t.dtype != dtype or t.dim() != dim or not t.is_contiguous():
            return None
    rows, hidden, head_dim = ids.shape[0], table.shape[1], cos_table.shape[1]
    if rows == 0 or positions.shape != ids.shape or sin_table.shape != cos_table.shape or hidden % 8 or head_dim % 8 \
            or not hidden or not head_dim or 0 in table.shape or 0 in cos_table.shape:
        return None
    if any(t.data_ptr() % 16 for t in (table, cos_table, sin_table)):
        return None
    out = torch.empty(rows, hidden, device=ids.device, dtype=torch.bfloat16)
    cos = torch.empty(rows, head_dim, device=ids.device, dtype=torch.bfloat16)
    sin = torch.empty_like(cos)
    rc = _lib.lib().bvllm_embed_rows(ids.data_ptr(), table.data_ptr(), table.shape[0], out.data_ptr(),
                                     positions.data_ptr(), cos_table.data_ptr(), sin_table.data_ptr(),
                                     cos_table.shape[0], cos.data_ptr(), sin.data_ptr(), rows, hidden, head_dim,
                                     stream)
    _lib.check(rc, "bvllm_embed_rows")
    return out, cos, sin
