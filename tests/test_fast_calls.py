"""The wrappers' native host side (csrc/fast_calls.cpp): its plan equals decode_split_plan, it declines
what it must decline, and calls through it equal calls through the Python path."""

import random

import pytest
import torch

from tests._cases import build_prefill_case, make_decode_inputs, python_path



def _fast():
    from babyvllm.kernels import _lib

    return _lib.fast()


def test_auto_plan_equals_decode_split_plan(monkeypatch):
    from babyvllm.kernels import decode_split as ds

    monkeypatch.delenv(ds.DECODE_PARTITION_ENV, raising=False)
    r = random.Random(4)
    for _ in range(3000):
        batch, hkv, width = r.randint(1, 300), r.choice([1, 2, 4, 8, 28]), r.choice([0, 1, 2, 129, r.randint(1, 5000)])
        max_len = r.choice([None, 0, 1, 16, 17, r.randint(0, 90000)])
        cus = r.choice([1, 132, 256, 304])
        got = _fast().auto_plan(batch, hkv, 16, width, -1 if max_len is None else max_len, cus, ds.MIN_PARTITION_BLOCKS)
        assert got == ds.decode_split_plan(batch, hkv, 16, width, max_len, cus), (batch, hkv, width, max_len, cus)


def test_auto_plan_at_the_ends_of_the_integers(monkeypatch):
    import sys

    from babyvllm.kernels import decode_split as ds

    monkeypatch.delenv(ds.DECODE_PARTITION_ENV, raising=False)
    for batch, width in ((1, 2048), (8, 130), (64, 300), (3, 1)):
        for max_len in (sys.maxsize - 15, sys.maxsize - 14, sys.maxsize, 2 ** 63, 2 ** 80):
            want = ds.decode_split_plan(batch, 4, 16, width, max_len, 256)
            assert _fast().auto_plan(batch, 4, 16, width, max_len, 256, ds.MIN_PARTITION_BLOCKS) == want, (batch, max_len)


def test_auto_plan_declines_a_page_size_it_cannot_divide_by():
    import subprocess
    import sys
    from pathlib import Path

    pkg = Path(__file__).resolve().parents[1] / "baby-vllm_amd"
    code = (f"import sys; sys.path.insert(0, {str(pkg)!r}); from babyvllm.kernels import _lib\n"
            "assert _lib.fast().auto_plan(1, 4, 0, 8, 100, 256, 4) is None")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, (out.returncode, out.stderr)


def test_cpu_tensors_and_wrong_argument_counts_are_declined():
    x = torch.zeros(2, 8, dtype=torch.bfloat16)
    f = _fast()
    assert f.norm(x, None, x[0], 1e-6, 0, 0) is None
    assert f.silu(x, 0, 0) is None
    assert f.linear(x, x, None, None, False, False, 0, 0) is None
    assert f.norm() is None and f.decode(x) is None and f.prefill() is None and f.rope(x, x) is None


@pytest.mark.parametrize("version", [None, 1])
def test_a_module_of_another_abi_is_refused(version, monkeypatch):
    import types

    import babyvllm
    from babyvllm.kernels import _lib

    assert _fast().ABI_VERSION == _lib.ABI_VERSION
    bound = []
    stale = types.SimpleNamespace(__file__="stale.so", names=_fast().names, bind=lambda *a: bound.append(a))
    if version is not None:
        stale.ABI_VERSION = version
    monkeypatch.setattr(babyvllm, "_fast_calls", stale)
    with pytest.raises(_lib.KernelLibraryError, match="rebuild"):
        _lib.fast.__wrapped__()
    assert not bound


def test_the_module_loads_in_a_process_that_has_not_imported_torch():
    import subprocess
    import sys
    from pathlib import Path

    pkg = Path(__file__).resolve().parents[1] / "baby-vllm_amd"
    code = f"import sys; sys.path.insert(0, {str(pkg)!r}); from babyvllm.kernels import _lib; _lib.fast()"
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr


def _calls():
    from babyvllm.kernels.activation import fused_silu_mul
    from babyvllm.kernels.layernorm import fused_add_rms_norm
    from babyvllm.kernels.paged_attn import paged_decode_attention
    from babyvllm.kernels.paged_prefill import paged_prefill_attention
    from babyvllm.kernels.rope import fused_rope_and_cache

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(sum(shape)))

    x, res = rand(3, 5, 96).bfloat16(), rand(3, 5, 96).bfloat16()
    out = {}
    for w in (rand(96), rand(96).bfloat16()):
        for r in (None, res.clone()):
            out["norm", w.dtype, r is None] = (fused_add_rms_norm(x, r, w, 1e-5), r)
    out["norm view"] = fused_add_rms_norm(rand(4, 200).bfloat16()[:, :96], None, rand(96), 1e-5)
    out["silu"] = fused_silu_mul(x)
    qkv = rand(7, 14 * 64 + 4 * 64).bfloat16()
    q, k, v = qkv[:, :896].view(7, 14, 64), qkv[:, 896:1024].view(7, 2, 64), qkv[:, 1024:].view(7, 2, 64)
    cache = rand(2, 4, 16, 2, 64).bfloat16()
    slots = torch.tensor([3, 60, 17, 9, 31, -1, 40], device="cuda")
    cos, sin = rand(7, 64).bfloat16(), rand(7, 64).bfloat16()
    fused_rope_and_cache(q, k, v, cos, sin, cache, slots)
    out["rope"] = (qkv, cache)
    for lens in ([40, 700, 0], [3000] + [20] * 39):
        dq, dc, bt, sl = make_decode_inputs(lens)
        for bucket in (None, max(lens), 4096):
            out["decode", len(lens), bucket] = paged_decode_attention(dq, dc, bt, sl, 0.1, max_seq_len=bucket)
    for specs in ([(0, 20), (30, 1), (5, 70)], [(5000, 40), (3000, 7)], [(0, 50), (4000, 1), (9, 1), (20, 1)],
                  [(6000, 40), (3000, 1), (40, 7), (70, 1), (9, 1)]):
        pq, pc, md = build_prefill_case(specs, 4, 7, 128)
        out["prefill", str(specs)] = paged_prefill_attention(pq, pc, md, 0.1)
    return out


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
def test_calls_equal_the_python_path(monkeypatch):
    native = _calls()
    python_path(monkeypatch)
    python = _calls()
    assert native.keys() == python.keys()
    for name in native:
        a, b = native[name], python[name]
        for s, t in zip(a if isinstance(a, tuple) else (a,), b if isinstance(b, tuple) else (b,)):
            assert (s is None) == (t is None), name
            if s is not None:
                assert s.shape == t.shape and s.dtype == t.dtype and s.stride() == t.stride(), name
                assert torch.equal(s, t), name


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("max_len", [-5, 2 ** 63 - 1, 2 ** 63, 2 ** 70, -2 ** 70])
def test_decode_takes_a_bucket_of_any_size_as_the_python_path_does(max_len, monkeypatch):
    from babyvllm.kernels.paged_attn import paged_decode_attention

    args = make_decode_inputs([900, 40, 0])
    native = paged_decode_attention(*args, 0.1, max_seq_len=max_len)
    python_path(monkeypatch)
    assert torch.equal(native, paged_decode_attention(*args, 0.1, max_seq_len=max_len))


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("path", ["native", "python"])
@pytest.mark.parametrize("op", ["decode", "prefill", "linear"])
def test_calls_without_the_memory_for_scratch_take_the_form_that_needs_none(op, path, monkeypatch):
    """A serving process may have given the card to its KV pool: calls that ran without scratch
    before they had a faster form with some still run."""
    import babyvllm.kernels.paged_prefill as pp
    from babyvllm.kernels.paged_attn import paged_decode_attention
    from babyvllm.layers.linear import Linear

    if path == "python":
        python_path(monkeypatch)
    if op == "decode":
        args = make_decode_inputs([9000] + [40] * 39)
        call = lambda: paged_decode_attention(*args, 0.1)
        plain = lambda: paged_decode_attention(*args, 0.1, partition_blocks=0)
    elif op == "prefill":
        args = build_prefill_case([(6000, 150)], 4, 7, 128)
        call = lambda: pp.paged_prefill_attention(*args, 0.1)

        def plain():
            with monkeypatch.context() as m:
                python_path(m)
                m.setattr(pp, "_split_tiles", lambda *a: 0)
                return pp.paged_prefill_attention(*args, 0.1)
    else:
        lin = Linear(18944, 3584, bias=False).to("cuda", torch.bfloat16)
        x = torch.randn(64, 18944, device="cuda", dtype=torch.bfloat16)
        call = lambda: lin(x)
        plain = lambda: torch.nn.functional.linear(x, lin.weight)
    with torch.no_grad():
        want, usual = plain(), call()
        assert path == "python" and op == "linear" or not torch.equal(want, usual)  # (sums in another order)
        del usual
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        out = torch.empty_like(want)
        total = torch.cuda.get_device_properties(0).total_memory
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        try:
            rest = []  # all that is left of the reserved memory, but for the output's block
            for size in (1 << 30, 1 << 26, 1 << 23, 1 << 21, 1100000):
                while True:
                    try:
                        rest.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
                    except torch.OutOfMemoryError:
                        break
            del out
            got = call()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
def test_refused_calls_raise_as_before():
    from babyvllm.kernels._lib import KernelLibraryError
    from babyvllm.kernels.activation import fused_silu_mul
    from babyvllm.kernels.layernorm import fused_add_rms_norm
    from babyvllm.kernels.paged_attn import paged_decode_attention
    from babyvllm.kernels.paged_prefill import paged_prefill_attention

    x = torch.randn(4, 96, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(TypeError):
        fused_add_rms_norm(x.float(), None, x[0], 1e-5)
    with pytest.raises(TypeError):
        fused_add_rms_norm(x, x[:, :8].contiguous(), x[0], 1e-5)
    with pytest.raises(RuntimeError):  # .view of a non-contiguous input
        fused_add_rms_norm(x.view(2, 2, 96).transpose(0, 1), None, x[0], 1e-5)
    with pytest.raises(AssertionError):
        fused_silu_mul(x[:, :32])
    q, cache, bt, lens = make_decode_inputs([20, 30])
    with pytest.raises(TypeError):
        paged_decode_attention(q, cache, bt.long(), lens, 0.1)
    with pytest.raises(ValueError):
        paged_decode_attention(q, cache, bt[:1], lens, 0.1)
    q96, cache96 = q[..., :96].contiguous(), cache[..., :96].contiguous()
    with pytest.raises(KernelLibraryError):  # head_dim the library refuses
        paged_decode_attention(q96, cache96, bt, lens, 0.1)
    pq, pc, md = build_prefill_case([(0, 5)], 4, 7, 128)
    with pytest.raises(AssertionError):
        paged_prefill_attention(pq[..., :96].contiguous(), pc, md, 0.1)
    for page, buckets in ((0, (None, 40)), (8, (None, 40))):  # pages of another size than 16 tokens
        for bucket in buckets:
            with pytest.raises((KernelLibraryError, ZeroDivisionError)):
                paged_decode_attention(q, cache[:, :, :page].contiguous(), bt, lens, 0.1, max_seq_len=bucket)
        with pytest.raises(KernelLibraryError):
            paged_prefill_attention(pq, pc[:, :, :page].contiguous(), md, 0.1)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("op", ["norm", "rope"])
def test_writes_to_a_lazy_clone_leave_its_source_alone(op):
    from babyvllm.kernels.layernorm import fused_add_rms_norm
    from babyvllm.kernels.rope import fused_rope_and_cache

    def rand(*shape):
        return torch.randn(*shape, device="cuda").bfloat16()

    if op == "norm":
        sources = [rand(4, 96)]
        x, w = rand(4, 96), rand(96)
    else:
        sources = [rand(3, 4, 64), rand(3, 2, 64), rand(2, 4, 16, 2, 64)]
        v, cos, sin, slots = rand(3, 2, 64), rand(3, 64), rand(3, 64), torch.tensor([5, 20, 40], device="cuda")

    def call(written):
        if op == "norm":
            fused_add_rms_norm(x, written[0], w, 1e-5)
        else:
            fused_rope_and_cache(written[0], written[1], v, cos, sin, written[2], slots)
        return written

    expected = call([s.clone() for s in sources])
    before = [s.clone() for s in sources]
    got = call([torch._lazy_clone(s) for s in sources])
    for s, b, g, e in zip(sources, before, got, expected):
        assert torch.equal(s, b) and torch.equal(g, e) and not torch.equal(g, b)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")
@pytest.mark.parametrize("op", ["norm", "silu", "rope", "decode", "prefill", "linear"])
def test_an_error_code_after_the_launch_raises_and_nothing_runs_twice(op, monkeypatch):
    """A code left behind by an earlier failed call comes back from a launch that ran:
    the call raises, the in-place kernels have run once and no other path is taken."""
    import ctypes

    from babyvllm.kernels import _lib
    from babyvllm.kernels.activation import fused_silu_mul
    from babyvllm.kernels.layernorm import fused_add_rms_norm
    from babyvllm.kernels.paged_attn import paged_decode_attention
    from babyvllm.kernels.paged_prefill import paged_prefill_attention
    from babyvllm.kernels.rope import fused_rope_and_cache
    from babyvllm.layers.linear import Linear

    def rand(*shape):
        return torch.randn(*shape, device="cuda").bfloat16()

    x, w = rand(4, 256), rand(256)
    if op == "norm":
        name, state = "bvllm_fused_add_rms_norm", [rand(4, 256)]
        call = lambda s: fused_add_rms_norm(x, s[0], w, 1e-5)
    elif op == "silu":
        name, state, call = "bvllm_silu_mul", [], lambda s: fused_silu_mul(x)
    elif op == "rope":
        v, cos, sin, slots = rand(3, 2, 64), rand(3, 64), rand(3, 64), torch.tensor([5, 20, 40], device="cuda")
        name, state = "bvllm_rope_kv_append", [rand(3, 4, 64), rand(3, 2, 64), rand(2, 4, 16, 2, 64)]
        call = lambda s: fused_rope_and_cache(s[0], s[1], v, cos, sin, s[2], slots)
    elif op == "decode":
        args = make_decode_inputs([20, 30])
        name, state, call = "bvllm_paged_decode", [], lambda s: paged_decode_attention(*args, 0.1)
    elif op == "prefill":
        args = build_prefill_case([(0, 5)], 4, 7, 128)
        name, state, call = "bvllm_paged_prefill", [], lambda s: paged_prefill_attention(*args, 0.1)
    else:
        lin = Linear(256, 64).to("cuda", torch.bfloat16)
        name, state, call = "bvllm_linear", [], lambda s: lin(x)
    with torch.no_grad():
        once = [t.clone() for t in state]
        call(once)
        fast, handle = _lib.fast(), _lib.lib()
        real, calls = getattr(handle, name), []

        def runs_and_fails(*a):
            calls.append(real(*a))
            return 1

        stub = ctypes.CFUNCTYPE(real.restype, *real.argtypes)(runs_and_fails)
        addresses = {n: ctypes.cast(getattr(handle, n), ctypes.c_void_p).value for n in fast.names()}
        try:
            fast.bind({**addresses, name: ctypes.cast(stub, ctypes.c_void_p).value}, _lib.check)
            with pytest.raises(_lib.KernelLibraryError, match=name):
                call(state)
        finally:
            fast.bind(addresses, _lib.check)
        assert calls == [0]
        for got, want in zip(state, once):
            assert torch.equal(got, want)
