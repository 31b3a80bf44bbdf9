"""nn.Linear whose few-token calls run on the HIP kernel (babyvllm/models/qwen2.py:17-137).

Same parameters, state dict and hooks as ``nn.Linear``; a call that is not one for
the kernel (more rows, autograd, tracing, other types or devices) is ``nn.Linear``'s.
"""

from __future__ import annotations

import torch.nn as nn

from babyvllm.kernels.linear import skinny_linear


class Linear(nn.Linear):
    def forward(self, x):
        y = skinny_linear(x, self.weight, self.bias)
        return super().forward(x) if y is None else y
