"""Linear layers of a few tokens (bvllm_linear): values against float64, and which calls torch keeps."""

import pytest
import torch

from tests._cases import assert_linear_close

pytestmark = pytest.mark.gpu

# (tokens, columns, k, gated): token-tile edges; columns that are no multiple of a
# row tile or of the split's unit; one stage of k, slabs of unequal length, k split
# over work-groups, and each wave layout of the launch rule.
SHAPES = [
    (1, 64, 128, False), (3, 100, 384, False), (16, 1152, 896, False), (17, 1156, 896, False),
    (64, 896, 896, False), (5, 2564, 640, False), (16, 4608, 3584, False), (32, 4600, 1152, False),
    (33, 4608, 3584, False), (1, 32772, 256, False), (16, 33000, 896, False), (32, 65540, 640, False),
    (48, 65536, 1024, False), (64, 65540, 256, False),
    (2, 896, 8192, False), (16, 900, 18944, False), (33, 3584, 8320, False), (64, 260, 18944, False),
    (24, 896, 4864, False), (64, 896, 4864, False),
    (65, 900, 10240, False), (128, 3584, 8192, False), (129, 260, 18944, False), (200, 896, 17408, False),
    (256, 3584, 18944, False),
    (1, 64, 128, True), (16, 4864, 896, True), (33, 4868, 896, True), (64, 8192, 384, True), (64, 8196, 384, True),
    (16, 18944, 3584, True), (17, 9000, 640, True),
    (65, 4864, 896, True), (97, 8964, 1536, True), (128, 64, 128, True), (129, 4868, 896, True), (192, 4864, 896, True),
    (256, 4864, 896, True), (65, 896, 4864, False), (65, 3588, 6272, False), (96, 3588, 3584, False), (128, 5120, 3584, False),
]


@pytest.mark.parametrize("m,n,k,gated", SHAPES)
def test_values_against_float64(m, n, k, gated):
    from babyvllm.kernels.linear import gated_linear, skinny_linear

    buf = torch.randn(m, k + 8, device="cuda", dtype=torch.bfloat16)
    x = buf[:, :k]  # a strided view
    w = torch.randn(n * (2 if gated else 1), k, device="cuda", dtype=torch.bfloat16) * 0.05
    bias = None if gated else torch.randn(n, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        got = gated_linear(x, w) if gated else skinny_linear(x, w, bias)
    assert got is not None and got.shape == (m, n)
    assert_linear_close(got, x, w, bias, gated)


def test_a_captured_call_takes_the_faster_kernel_on_the_gpu():
    """Some shapes beyond 64 tokens save an eager caller the library's host time; a captured step
    pays none, and there the library's GEMM ends sooner."""
    from babyvllm.kernels.linear import gated_linear, skinny_linear

    x = torch.randn(160, 896, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(2 * 4864, 896, device="cuda", dtype=torch.bfloat16)
    y = torch.randn(96, 4864, device="cuda", dtype=torch.bfloat16)
    v = torch.randn(896, 4864, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        assert gated_linear(x, w) is not None and skinny_linear(y, v) is not None
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = gated_linear(x, w), skinny_linear(y, v), gated_linear(x[:128], w)
        assert captured[0] is None and captured[1] is None and captured[2] is not None


def test_same_bits_for_any_batch_of_a_token_tile_count_and_in_a_graph():
    from babyvllm.kernels.linear import skinny_linear

    x = torch.randn(16, 8192, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(896, 8192, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        full = skinny_linear(x, w)
        for m in (1, 7, 16):
            assert torch.equal(skinny_linear(x[:m], w), full[:m])
        out = torch.empty_like(full)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            skinny_linear(x, w, None, out)
        for scale in (1.0, -2.0, 0.5):
            x.mul_(scale)
            graph.replay()
            assert torch.equal(out, skinny_linear(x, w))


def test_out_is_an_in_place_write_to_autograd():
    """As torch.mm(..., out=): the version moves, a backward through overwritten values and a
    write to an inference tensor outside inference mode raise."""
    from babyvllm.kernels.linear import skinny_linear

    x = torch.randn(4, 256, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(64, 256, device="cuda", dtype=torch.bfloat16)
    out = torch.randn(4, 64, device="cuda", dtype=torch.bfloat16)
    scale = torch.ones(64, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    loss = (out * scale).sum()
    version = out._version
    with torch.no_grad():
        assert skinny_linear(x, w, None, out) is not None
    assert out._version == version + 1
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()
    with torch.inference_mode():
        inference = torch.zeros(4, 64, device="cuda", dtype=torch.bfloat16)
        assert skinny_linear(x, w, None, inference) is not None
        kept = inference.clone()
        assert skinny_linear(x, w, None, out) is not None
    with torch.no_grad(), pytest.raises(RuntimeError, match="inference tensor"):
        skinny_linear(x + 1, w, None, inference)
    assert torch.equal(inference, kept)


def test_non_finite_weights_and_inputs_stay_in_their_row_and_column():
    from babyvllm.kernels.linear import skinny_linear

    x = torch.randn(5, 640, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(68, 640, device="cuda", dtype=torch.bfloat16)
    w[67, 639], w[3, 0], x[4, 7] = float("inf"), float("nan"), float("nan")
    with torch.no_grad():
        got = skinny_linear(x, w)
    want = x.double() @ w.double().T
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())


def test_module_keeps_autograd_hooks_and_other_types():
    from babyvllm.kernels.linear import gated_linear, skinny_linear
    from babyvllm.layers.linear import Linear
    from babyvllm.models.qwen2 import Qwen2MLP

    lin = Linear(256, 64).to("cuda", torch.bfloat16)
    ref = torch.nn.Linear(256, 64).to("cuda", torch.bfloat16)
    ref.load_state_dict(lin.state_dict())
    x = torch.randn(4, 256, device="cuda", dtype=torch.bfloat16)
    assert skinny_linear(x, lin.weight, lin.bias) is None  # grad mode: torch's operation
    lin(x).sum().backward()
    ref(x).sum().backward()
    assert torch.equal(lin.weight.grad, ref.weight.grad)
    with torch.no_grad():
        assert skinny_linear(x, lin.weight, lin.bias) is not None
        assert skinny_linear(x.float(), lin.weight.float()) is None
        assert skinny_linear(x[:, ::2], lin.weight[:, :128].contiguous()) is None
        assert skinny_linear(x[:1].expand(4, 256), lin.weight) is None
        assert skinny_linear(torch.randn(65, 256, device="cuda", dtype=torch.bfloat16), lin.weight) is None
        with torch.autocast("cuda", dtype=torch.float16):
            assert skinny_linear(x, lin.weight, lin.bias) is None and lin(x).dtype == torch.float16
        batched = torch.func.vmap(lambda r: lin(r))(x.view(4, 1, 256))
        torch.testing.assert_close(batched.view(4, 64), ref(x), atol=2e-2, rtol=2e-2)

        mlp = Qwen2MLP(256, 128).to("cuda", torch.bfloat16)
        fused = mlp(x)
        seen = []
        hook = mlp.gate_up_proj.register_forward_hook(lambda m, i, o: seen.append(o))
        torch.testing.assert_close(mlp(x), fused, atol=2e-3, rtol=2e-2)
        hook.remove()
        assert len(seen) == 1 and seen[0].shape == (4, 256)
        assert gated_linear(x, mlp.gate_up_proj.weight) is not None


# ------------------------------------------------------------------ input rows


@pytest.mark.parametrize("rows,hidden,dim", [(1, 8, 8), (3, 896, 64), (16, 3584, 128), (65, 264, 72), (700, 3584, 128)])
def test_embed_rows_equals_torch(rows, hidden, dim):
    from babyvllm.kernels.embed import embed_rows

    table = torch.randn(50, hidden, device="cuda", dtype=torch.bfloat16)
    cos, sin = torch.randn(40, dim, device="cuda"), torch.randn(40, dim, device="cuda")
    ids = torch.randint(0, 50, (rows,), device="cuda")
    pos = torch.randint(-40, 40, (rows,), device="cuda")
    with torch.no_grad():
        got = embed_rows(ids, table, pos, cos, sin)
    for a, b in zip(got, (table[ids], cos[pos].bfloat16(), sin[pos].bfloat16())):
        assert torch.equal(a, b) and a.dtype == b.dtype
    with torch.no_grad():  # outside the tables: NaN rows, the others untouched
        ids[0], pos[-1] = 50, 40
        h, c, s = embed_rows(ids, table, pos, cos, sin)
    assert h[0].isnan().all() and c[-1].isnan().all() and s[-1].isnan().all()
    assert torch.equal(h[1:], table[ids[1:]])


def test_model_input_rows_keep_hooks_and_modules():
    from babyvllm.config import ModelConfig
    from babyvllm.models.qwen2 import Qwen2Model

    cfg = ModelConfig(vocab_size=40, hidden_size=128, intermediate_size=256, num_hidden_layers=0,
                      num_attention_heads=2, num_key_value_heads=1, rms_norm_eps=1e-6, max_position_embeddings=64,
                      rope_theta=1e4, tie_word_embeddings=True)
    model = Qwen2Model(cfg).to("cuda")
    model.embed_tokens.to(torch.bfloat16)
    ids, pos = torch.tensor([3, 39, 0], device="cuda"), torch.tensor([0, 63, 5], device="cuda")
    with torch.no_grad():
        one = model._input_rows(ids, pos)
        seen = []
        hook = model.embed_tokens.register_forward_hook(lambda m, i, o: seen.append(o))
        two = model._input_rows(ids, pos)
        hook.remove()
    assert len(seen) == 1
    for a, b in zip(one, two):
        assert torch.equal(a, b) and a.dtype == b.dtype
    assert model._input_rows(ids, pos)[0].requires_grad  # grad mode: torch's operations
