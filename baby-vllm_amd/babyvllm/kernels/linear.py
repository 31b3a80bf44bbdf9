"""Linear layers of a few tokens on the HIP kernel (the nn.Linear calls of babyvllm/models/qwen2.py:17-137).

``skinny_linear(x, weight, bias, out)`` and ``gated_linear(x, weight)`` compute a
decode step's linear layers (and an MLP's fused gate/up projection with SiLU·mul)
with ``bvllm_linear`` and return the result, or return ``None`` when the call is not
one for that kernel; the caller then takes torch's own operations. The kernel takes
plain bf16 tensors of at most 64 rows on the current ROCm device, outside autograd
and outside every mode that has to see torch operations (tracing, compilation,
functorch transforms, forward-mode AD, dispatch and function modes, autocast).
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad

from babyvllm.kernels import _lib

MAX_ROWS = 64


def _torch_must_see(*tensors) -> bool:
    """Whether something besides the values wants to see this operation."""
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors):
        return True
    c = torch._C
    return (c._len_torch_dispatch_stack() > 0 or c._len_torch_function_stack() > 0
            or c._functorch.peek_interpreter_stack() is not None or forward_ad._current_level >= 0
            or c._get_tracing_state() is not None or torch.compiler.is_compiling()
            or torch.is_autocast_enabled("cuda"))


def _plain(t, dtype) -> bool:
    return type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda and t.dtype == dtype


def _launch(x, weight, bias, out, n, gated):
    rows, k = x.shape
    if k != weight.shape[1] or x.device != weight.device or x.device.index != torch.cuda.current_device():
        return None
    if x.stride(1) != 1 or not weight.is_contiguous():
        return None
    x_stride = x.stride(0) if rows > 1 else k
    if x_stride < k or x_stride % 8 or x.data_ptr() % 16 or weight.data_ptr() % 16:
        return None
    if bias is not None and not (_plain(bias, torch.bfloat16) and bias.device == x.device and bias.is_contiguous()
                                 and bias.shape == (n,)):
        return None
    if out is None:
        out = torch.empty(rows, n, device=x.device, dtype=torch.bfloat16)
    elif not (_plain(out, torch.bfloat16) and out.device == x.device and out.shape == (rows, n)
              and out.stride(1) == 1 and (rows == 1 or out.stride(0) >= n and out.stride(0) % 4 == 0)
              and out.data_ptr() % 8 == 0):
        return None
    h = _lib.lib()
    nbytes = h.bvllm_linear_workspace_bytes(rows, n, k, gated)
    if nbytes < 0:
        return None
    workspace = torch.empty(nbytes // 4, device=x.device, dtype=torch.float32) if nbytes else None
    rc = h.bvllm_linear(x.data_ptr(), x_stride, weight.data_ptr(), None if bias is None else bias.data_ptr(),
                        out.data_ptr(), out.stride(0) if rows > 1 else n, rows, n, k, gated,
                        None if workspace is None else workspace.data_ptr(), _lib.stream_handle(x.device))
    _lib.check(rc, "bvllm_linear")
    return out


def skinny_linear(x, weight, bias=None, out=None):
    """``x @ weight.T + bias`` for x [M ≤ 64, K] (into ``out`` if given), or None."""
    if x.dim() != 2 or weight.dim() != 2 or not 0 < x.shape[0] <= MAX_ROWS:
        return None
    if not (_plain(x, torch.bfloat16) and _plain(weight, torch.bfloat16)) or _torch_must_see(x, weight, bias, out):
        return None
    return _launch(x, weight, bias, out, weight.shape[0], 0)


def gated_linear(x, weight):
    """``silu(x @ gate.T) * (x @ up.T)`` for weight = [gate; up], x [M ≤ 64, K], or None.

    Gate and up stay fp32 up to the product (torch's two steps round them to bf16 first).
    """
    if x.dim() != 2 or weight.dim() != 2 or weight.shape[0] % 2 or not 0 < x.shape[0] <= MAX_ROWS:
        return None
    if not (_plain(x, torch.bfloat16) and _plain(weight, torch.bfloat16)) or _torch_must_see(x, weight):
        return None
    return _launch(x, weight, None, None, weight.shape[0] // 2, 1)
