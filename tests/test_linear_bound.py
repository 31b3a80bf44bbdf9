"""The check of the linear kernel's values fails for a sum with a part missing (float arithmetic on the CPU)."""

import pytest
import torch
import torch.nn.functional as F

from tests._cases import assert_linear_close


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("missing", [0, 16])
def test_a_missing_slice_of_k_is_seen(gated, missing):
    m, n, k = 16, 500, 3584
    x = torch.randn(m, k).bfloat16()
    w = (torch.randn(n * (2 if gated else 1), k) * 0.05).bfloat16()
    seen = x.clone()
    seen[:, k - missing:] = 0
    y = seen.float() @ w.float().T
    got = (F.silu(y[:, :n]) * y[:, n:] if gated else y).bfloat16()
    if missing:
        with pytest.raises(AssertionError):
            assert_linear_close(got, x, w, None, gated)
    else:
        assert_linear_close(got, x, w, None, gated)
