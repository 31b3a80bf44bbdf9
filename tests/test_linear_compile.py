"""Projections under torch.compile: traced whole, as nn.Linear is."""

import pytest
import torch


def test_what_torch_must_see_is_asked_without_a_graph_break():
    from babyvllm.kernels.linear import torch_must_see

    def f(x, w):
        return x @ w.T if torch_must_see(x, w) else x

    x, w = torch.randn(4, 8), torch.randn(3, 8)
    assert not torch_must_see(x, w)
    torch._dynamo.reset()
    assert torch.equal(torch.compile(f, backend="eager", fullgraph=True)(x, w), x @ w.T)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("grad", [False, True])
def test_linear_compiles_in_one_graph(grad):
    from babyvllm.layers.linear import Linear

    lin = Linear(256, 64).to("cuda", torch.bfloat16)
    ref = torch.nn.Linear(256, 64).to("cuda", torch.bfloat16)
    ref.load_state_dict(lin.state_dict())
    x = torch.randn(4, 256, device="cuda", dtype=torch.bfloat16)
    torch._dynamo.reset()
    with torch.set_grad_enabled(grad):
        got = torch.compile(lin, backend="eager", fullgraph=True)(x)
        assert torch.equal(got, ref(x)) and got.requires_grad == grad
