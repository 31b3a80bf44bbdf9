"""Linear layers of a few tokens on the HIP kernel (the nn.Linear calls of babyvllm/models/qwen2.py:17-137).

``skinny_linear(x, weight, bias, out)`` and ``gated_linear(x, weight)`` compute a
decode step's linear layers (and an MLP's fused gate/up projection with SiLU·mul)
with ``bvllm_linear`` and return the result, or return ``None`` when the call is not
one for that kernel; the caller then takes torch's own operations. The kernel takes
plain bf16 tensors of at most 256 rows, of the shapes where it ends sooner than a
library GEMM (``bvllm_linear_workspace_bytes``), on the current ROCm device, outside autograd and outside every mode
that has to see torch operations (tracing, compilation, functorch transforms,
forward-mode AD, dispatch and function modes, autocast).
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad

from babyvllm.kernels import _lib

MAX_ROWS = 256


def torch_must_see(*tensors) -> bool:
    """Whether something besides the values wants to see this operation."""
    if torch.compiler.is_compiling():  # first: the questions below are none the compiler can trace
        return True
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors):
        return True
    c = torch._C
    return (c._len_torch_dispatch_stack() > 0 or c._len_torch_function_stack() > 0
            or c._functorch.peek_interpreter_stack() is not None or forward_ad._current_level >= 0
            or c._get_tracing_state() is not None or torch.is_autocast_enabled("cuda"))


def _eager(x) -> bool:
    """Whether the library's host time counts: a captured step pays none (up to 64 rows the kernel's
    choice does not ask)."""
    return x.shape[0] > 64 and not torch.cuda.is_current_stream_capturing()


def skinny_linear(x, weight, bias=None, out=None):
    """``x @ weight.T + bias`` for x [M, K] (into ``out`` if given), or None."""
    if not x.is_cuda or x.dim() != 2 or x.shape[0] > MAX_ROWS or torch_must_see(x, weight, bias, out):
        return None
    return _lib.fast().linear(x, weight, bias, out, False, _eager(x), *_lib.current())


def gated_linear(x, weight):
    """``silu(x @ gate.T) * (x @ up.T)`` for weight = [gate; up], x [M, K], or None.

    Gate and up stay fp32 up to the product (torch's two steps round them to bf16 first).
    """
    if not x.is_cuda or x.dim() != 2 or x.shape[0] > MAX_ROWS or torch_must_see(x, weight):
        return None
    return _lib.fast().linear(x, weight, None, None, True, _eager(x), *_lib.current())
