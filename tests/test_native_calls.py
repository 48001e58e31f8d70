"""The native callers behind ops.py (csrc/torch_calls.cpp): the same results, bit for bit, as the Python below them, and None for what they leave
to it."""
import pytest


class _Declines:
    """Stands in for the extension module: every call is left to ops.py."""

    def __getattr__(self, name):
        return lambda *args: None


def _calls(ops, torch, dtype):
    """(name, call) pairs; a call may update tensors in place and returns every tensor that it wrote"""
    gen = torch.Generator(device="cuda")

    def rn(*shape):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, 1.0, generator=gen)

    gen.manual_seed(1)
    a, b, bn, bias = rn(9, 64), rn(64, 24), rn(24, 64), rn(24)
    padded, out = rn(9, 72)[:, :64], rn(12, 24)[:9]
    yield "mm", lambda: [ops.tensor_mm(a, b)]
    yield "mm nk", lambda: [ops.tensor_mm(padded, bn, b_layout=1)]
    yield "mm out", lambda: [ops.tensor_mm(a, b, out=out), out]
    yield "mm no rows", lambda: [ops.tensor_mm(a[:0], b)]
    if dtype == torch.float32:
        yield "mm a stored [K, M]", lambda: [ops.tensor_mm(bn.T.contiguous(), b, a_layout=1)]
    yield "gemm", lambda: [ops.tensor_gemm(a, b, bias)]
    yield "gemm nk", lambda: [ops.tensor_gemm(a, bn, bias, b_layout=1)]
    yield "softcap", lambda: [ops.tensor_gemma_linear_softcap(a.reshape(1, 9, 64), bn, 30)]
    yield "upproj", lambda: [ops.mlp_gemma2_fused_upproj(a.reshape(3, 3, 64), b, b.clone())]
    yield "upproj nk", lambda: [ops.mlp_gemma2_fused_upproj(a[0], bn, bn.clone(), b_layout=1)]
    yield "softmax", lambda: [ops.tensor_softmax(a, alpha=0.5, softcap=20.0, causal=True, window=7, q_len=3, diag=20)]
    yield "softmax out", lambda: [ops.tensor_softmax(padded, out=rn(9, 64))]
    yield "softmax int alpha", lambda: [ops.tensor_softmax(a, alpha=2)]
    x3, w4, bias9, state = rn(2, 9, 64), rn(9, 4), rn(9), rn(2, 9, 3)
    yield "conv1d", lambda: [ops.tensor_causal_conv1d(x3, w4, bias9)]
    yield "conv1d out", lambda: [ops.tensor_causal_conv1d(x3, w4, bias9, out=rn(2, 9, 64))]

    def update():
        s = state.clone()
        return [ops.tensor_causal_conv1d_update(x3[:, :, 0].contiguous(), s, w4, bias9), s]
    yield "conv1d update", update
    yield "conv1d update width 1", lambda: [ops.tensor_causal_conv1d_update(x3[:, :, 0].contiguous(), state[:, :, :0].contiguous(), w4[:, :1].contiguous(), bias9)]
    yield "rms norm", lambda: [ops.tensor_rms_norm(a, b[:, 0].contiguous(), 1e-5)]
    yield "gated norm", lambda: [ops.tensor_rms_norm(a, b[:, 0].contiguous(), 1e-5, True, padded.contiguous())]
    yield "gated norm of a group", lambda: [ops.tensor_zamba_gated_rmsnorm(x3, x3.clone(), a[0].contiguous(), 64, 1e-5)]
    q, k, v, mask = rn(1, 4, 20, 64), rn(1, 4, 50, 64), rn(1, 4, 50, 64), rn(1, 1, 20, 50)
    yield "masked", lambda: [ops.sdp_attention_masked_scaled_fwd(q, k, v, mask, 0.125)]
    yield "masked, dense after a copy", lambda: [ops.sdp_attention_masked_scaled_fwd(q, k, v, mask.expand(1, 1, 20, 50)[:, :, :, ::1], 0.125)]
    yield "masked, other head dimension", lambda: [ops.sdp_attention_masked_scaled_fwd(q[..., :32], k[..., :32], v[..., :32], mask, 0.125)]
    yield "attention", lambda: [ops.sdp_attention_fwd(q, k[:, :2], v[:, :2], 0.125, softcap=30.0, causal=True, window=16)]
    kl, vl = rn(1, 2, 300, 64), rn(1, 2, 300, 64)
    yield "attention, generation", lambda: [ops.sdp_attention_fwd(q[:, :, :2].contiguous(), kl, vl, 0.125, causal=True)]
    yield "attention, generation asked for", lambda: [ops.sdp_attention_fwd(q, kl, vl, 0.125, causal=True, decode=True)]
    yield "attention, generation refused", lambda: [ops.sdp_attention_fwd(q[:, :, :2].contiguous(), kl, vl, 0.125, causal=True, decode=False)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float16", "float32"])
def test_native_calls_give_the_bits_of_the_python_path(ops, monkeypatch, dtype):
    import torch
    first = {name: [t.clone() for t in call()] for name, call in _calls(ops, torch, getattr(torch, dtype))}
    monkeypatch.setattr(ops, "_native", _Declines())
    for name, call in _calls(ops, torch, getattr(torch, dtype)):
        for got, want in zip(first[name], call()):
            assert got.shape == want.shape and got.dtype == want.dtype and got.stride() == want.stride(), name
            assert torch.equal(got.reshape(-1).view(torch.uint8), want.reshape(-1).view(torch.uint8)), name


@pytest.mark.gpu
def test_native_calls_decline_what_they_do_not_check(ops):
    import torch
    from anygpu_amd import capi
    native = capi.load_torch_calls()
    a, b = torch.zeros(4, 8, device="cuda"), torch.zeros(8, 4, device="cuda")
    assert native.mm(a, b, None, 0, 0) is not None
    for args in ((a.cpu(), b, None, 0, 0), (a, b.half(), None, 0, 0), (a, a, None, 0, 0), (a.double(), b.double(), None, 0, 0), (a[:, ::2], b[:4], None, 0, 0),
                 (a, b, None, 2, 0), (a, b, None, 0, 2), (a.half(), b.half(), None, 0, 1), (a, b, torch.zeros(4, 5, device="cuda"), 0, 0), (None, b, None, 0, 0),
                 (a, b, None, 0.0, 0), (a, b, None, 1 << 80, 0)):
        assert native.mm(*args) is None
    seen = []

    def one(row):
        seen.append(native.softmax(row, None, 1.0, 0.0, False, 0, 0, 0))
        return row
    torch.vmap(one)(torch.zeros(3, 2, 4, device="cuda"))          # a wrapper whose class is Tensor
    assert seen == [None]
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with Mode():
        assert native.mm(a, b, None, 0, 0) is None
    # the C ABI's own refusal comes back as the package's error
    with pytest.raises(capi.AnyGpuError):
        native.softmax(a, None, 1.0, 0.0, False, -1, 0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,other", [("float32", "float16"), ("float16", "float32"), ("float32", "int32")])
def test_results_of_another_type_or_layout_are_refused(ops, dtype, other):
    # elements of the operands' type would run past the end of a narrower result, rows of a transposed one over each other
    import torch
    from anygpu_amd import capi
    native = capi.load_torch_calls()
    dtype, other = getattr(torch, dtype), getattr(torch, other)
    a, b, x = torch.zeros(4, 8, dtype=dtype, device="cuda"), torch.zeros(8, 6, dtype=dtype, device="cuda"), torch.zeros(2, 3, 8, dtype=dtype, device="cuda")
    mm_out, rows_out, conv_out = (torch.full(shape, 7, dtype=other, device="cuda") for shape in ((4, 6), (4, 8), (2, 3, 8)))
    w, bias = torch.zeros(3, 4, dtype=dtype, device="cuda"), torch.zeros(3, dtype=dtype, device="cuda")
    turned, turned_conv = torch.full((8, 4), 7, dtype=dtype, device="cuda").T, torch.full((2, 8, 3), 7, dtype=dtype, device="cuda").transpose(1, 2)
    assert native.mm(a, b, mm_out, 0, 0) is None and native.softmax(a, rows_out, 1.0, 0.0, False, 0, 0, 0) is None
    assert native.softmax(a, turned, 1.0, 0.0, False, 0, 0, 0) is None
    for call in (lambda: ops.tensor_mm(a, b, out=mm_out), lambda: ops.tensor_softmax(a, out=rows_out), lambda: ops.tensor_softmax(a, out=turned), lambda: ops.tensor_mm(a, b, out=mm_out.cpu()),
                 lambda: ops.tensor_softmax(a, out=rows_out.cpu()), lambda: ops.tensor_causal_conv1d(x, w, bias, out=conv_out), lambda: ops.tensor_causal_conv1d(x, w, bias, out=turned_conv)):
        with pytest.raises(ValueError):
            call()
    assert all(bool((t == 7).all()) for t in (mm_out, rows_out, conv_out, turned, turned_conv))


@pytest.mark.gpu
def test_a_dense_convolution_result_of_another_shape_takes_the_samples_in_order(ops):
    import torch
    x, w, bias = (torch.arange(n, dtype=torch.float32, device="cuda").reshape(shape) / n for n, shape in ((2 * 9 * 64, (2, 9, 64)), (9 * 4, (9, 4)), (9, (9,))))
    want = ops.tensor_causal_conv1d(x, w, bias)
    flat, larger = torch.full((18 * 64,), 7.0, device="cuda"), torch.full((20, 64), 7.0, device="cuda")
    assert ops.tensor_causal_conv1d(x, w, bias, out=flat) is flat and ops.tensor_causal_conv1d(x, w, bias, out=larger) is larger
    assert torch.equal(flat.view(2, 9, 64), want) and torch.equal(larger[:18].view(2, 9, 64), want) and bool((larger[18:] == 7).all())
    with pytest.raises(ValueError):
        ops.tensor_causal_conv1d(x, w, bias, out=flat[:-1])
    assert torch.equal(flat.view(2, 9, 64), want)


@pytest.mark.parametrize("content", [None, b"not a library"])
def test_without_the_extension_module_the_python_path_calls_the_library(monkeypatch, tmp_path, content):
    import torch
    from anygpu_amd import capi, ops
    path = tmp_path / "_torch_calls.so"
    if content is not None:
        path.write_bytes(content)
    monkeypatch.setattr(capi, "TORCH_CALLS_PATH", path)
    monkeypatch.setattr(ops, "_native", None)
    a = torch.zeros(2, 2)
    with pytest.warns(RuntimeWarning, match="ctypes"), pytest.raises(ValueError, match="device tensors only"):
        ops.tensor_mm(a, a)
    with pytest.raises(ValueError, match="device tensors only"):         # (the warning comes once)
        ops.tensor_softmax(a)
    monkeypatch.setattr(capi, "load", lambda: (_ for _ in ()).throw(RuntimeError("no library")))
    monkeypatch.setattr(ops, "_native", None)
    with pytest.raises(RuntimeError, match="no library"):                # there is no way around the library itself
        ops.tensor_mm(a, a)


def test_everything_but_the_extension_module_is_built_without_torch(monkeypatch):
    import importlib.util

    from anygpu_amd import build
    for name in ("build_kernels", "build_host_harness", "build_oracle", "build_torch_calls"):
        monkeypatch.setattr(build, name, lambda verbose, name=name: name)
    assert list(build.build_all().values()) == ["build_kernels", "build_host_harness", "build_oracle", "build_torch_calls"]
    find = importlib.util.find_spec
    monkeypatch.setattr(importlib.util, "find_spec", lambda name, *rest: None if name == "torch" else find(name, *rest))
    assert list(build.build_all().values()) == ["build_kernels", "build_host_harness", "build_oracle"]
