"""The torch operators' native kernels (csrc/torch_ops.cpp) against the Python functions that define
the operators: the same bits for ordinary calls, and everything else as the functions have it
(errors, empty tensors, autograd, tracing, vmap).  A call whose first tensor requires a gradient
runs the Python function."""
import os
import subprocess
import sys

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import __graft_entry__

B, L, H, D = 2, 37, 24, 128
C = H * D


def _calls(W, device, make):
    """name -> arguments, every operator with and without its optional tensors; make(shape, dtype)."""
    bf, f32 = torch.bfloat16, torch.float32
    qkv = make((B, L, 3 * C), bf)
    q, k, v = (t.unflatten(-1, (H, D)) for t in qkv.split(C, -1))
    kc, vc = make((B, 50, H, D), bf), make((B, 50, H, D), bf)
    long_ = [make((1, n, 2, D), bf) for n in (257, 1500, 1500)]       # a size with scratch
    g, cos, sin = make((C,), bf), make((L, 64), f32), make((L, 64), f32)
    lens = torch.tensor([50, 7], dtype=torch.int32, device=device)
    inv, sums = make((B, L), f32).abs(), make((4 * H, B * L), f32).abs() * 64
    x, y, e, e2 = make((B, L, C), bf), make((B, L, C), bf), make((1, 6, C), bf), make((1, 2, C), bf)
    w, b = make((512, 1024), bf), make((512,), bf)
    o = W.ops
    return {
        "flash_self_attn": (o.flash_self_attn, (q, k, v, 0.09, 0)),
        "flash_self_attn_part": (o.flash_self_attn, (*long_, 0.09, 1200)),
        "cross_attn": (o.cross_attn, (q, kc, vc, None, 0.09)),
        "cross_attn_lens": (o.cross_attn, (q, kc, vc, lens, 0.09)),
        "self_attn_fused": (o.self_attn_fused, (q, k, v, g, g, 1e-6, cos, sin, 0.09)),
        "self_attn_fused_sumsq": (o.self_attn_fused_sumsq, (q, k, v, sums, g, g, 1e-6, cos, sin, 0.09)),
        "cross_attn_fused": (o.cross_attn_fused, (q, kc, vc, g, 1e-6, None, 0.09)),
        "cross_attn_fused_lens": (o.cross_attn_fused, (q, kc, vc, g, 1e-6, lens, 0.09)),
        "flash_attn_qnorm": (o.flash_attn_qnorm, (q, k, v, inv, g, None, None, None, 0.09)),
        "flash_attn_qnorm_rope": (o.flash_attn_qnorm, (q, k, v, inv, g, cos, sin, None, 0.09)),
        "flash_attn_qnorm_lens": (o.flash_attn_qnorm, (q, kc, vc, inv, g, None, None, lens, 0.09)),
        "rope": (o.rope, (q, cos, sin)),
        "rms_norm": (o.rms_norm, (k, g, 1e-6)),
        "rms_norm_rope": (o.rms_norm, (k, g, 1e-6, cos, sin)),
        "rms_inv": (o.rms_inv, (k, 1e-6)),
        "adaln": (o.adaln_stage, (x, y, e, 1, 2, 0, 1, None, None, 1e-6, True)),
        "adaln_rows": (o.adaln_stage, (x, y, e, 1, 5, 0, 1, g, g, 1e-6, True, e2)),
        "adaln_norm": (o.adaln_stage, (x, None, None, 1, -1, -1, -1, None, None, 1e-6, True)),
        "adaln_gate": (o.adaln_stage, (x, y, e, 1, 2, -1, -1, None, None, 1e-6, False)),
        "qkv_proj_sumsq": (o.qkv_proj_sumsq, (make((B, L, 1024), bf), w, b, 256)),
        "qkv_proj": (o.qkv_proj_sumsq, (make((B, L, 1024), bf), w, b, 0)),
        "linear": (o.linear, (make((B, L, 1024), bf), w, b)),
    }


NAMES = list(_calls(type("W", (), {"ops": type("O", (), {"__getattr__": lambda s, n: None})()}), "cpu",
                    lambda shape, dtype: torch.zeros(shape, dtype=dtype)))


def _tuple(r):
    return r if isinstance(r, tuple) else (r,)


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_traces_on_fake_device_tensors(W):
    """The native autograd kernel hands fake tensors on to their mode, with and without gradients."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        for name, (op, args) in _calls(W, "cuda", lambda s, dtype: torch.empty(s, dtype=dtype, device="cuda")).items():
            for grad in (False, True):
                out = _tuple(op(args[0].detach().requires_grad_(grad), *args[1:]))
                assert out[0].device.type == "cuda" and out[0].requires_grad == grad, name


@pytest.mark.gpu
@pytest.mark.parametrize("name", NAMES)
def test_native_equals_python(W, name):
    gen = torch.Generator(device="cuda").manual_seed(3)
    make = lambda shape, dtype: torch.randn(shape, generator=gen, device="cuda").to(dtype)     # noqa: E731
    op, args = _calls(W, "cuda", make)[name]
    native = _tuple(op(*args))
    python = _tuple(op(args[0].detach().requires_grad_(), *args[1:]))
    for a, b in zip(native, python):
        assert not a.requires_grad and a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype
        if name == "qkv_proj" and a.dtype == torch.float32:
            continue                                            # no columns asked for: not written
        assert torch.equal(a, b.detach())
    needs = [t for t in python if t.requires_grad]
    assert needs
    with pytest.raises(RuntimeError, match="no autograd formula"):
        needs[0].sum().backward()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.inference_mode():
        again = _tuple(op(*args))
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(again[0], native[0])
    with _Seen() as seen:
        op(*args)
    assert any(s.startswith("wan_hip.") for s in seen.names)


@pytest.mark.gpu
@pytest.mark.parametrize("name", NAMES)
def test_none_for_a_tensor_is_told_by_the_function(W, name):
    """In place of every required tensor, the other arguments being ordinary ones: the Python function's
    error, never one about an undefined tensor."""
    op, args = _calls(W, "cuda", lambda shape, dtype: torch.zeros(shape, dtype=dtype, device="cuda"))[name]
    for i in [i for i, a in enumerate(op._opoverload._schema.arguments) if str(a.type) == "Tensor"]:
        with pytest.raises((TypeError, ValueError, AttributeError), match="None|must be a"):
            op(*args[:i], None, *args[i + 1:])


@pytest.mark.gpu
def test_other_calls_as_the_functions_have_them(W):
    o, dev = W.ops, "cuda"
    x = torch.randn(2, 5, 2, D, device=dev).bfloat16()
    g = torch.ones(2 * D, device=dev, dtype=torch.bfloat16)
    cos = torch.ones(5, 64, device=dev)
    for bad, what in ((x.float(), "bfloat16"), (x[..., :64], "head_dim"), (x[0], "expected"), (x.cpu(), "CUDA"),
                      (x.transpose(1, 3).contiguous().transpose(1, 3), "contiguous"),
                      (x.flatten()[1:1 + 4 * D].view(1, 2, 2, D), "aligned")):
        with pytest.raises(ValueError, match=what):
            o.rms_norm(bad, g, 1e-6)
    for args in ((x, g[1:], 1e-6), (x, g, 1e-6, cos), (x, g, 1e-6, cos, cos.double()), (x, g.cpu(), 1e-6)):
        with pytest.raises(ValueError):
            o.rms_norm(*args)
    with pytest.raises(ValueError, match="actual_seqlen_k"):
        o.flash_self_attn(x, x, x, 0.1, 6)
    with pytest.raises(ValueError, match="differ"):
        o.cross_attn(x, x, x[:, :3], None, 0.1)
    with pytest.raises(ValueError, match="seqlen_k"):
        o.cross_attn(x, x, x, torch.ones(2, device=dev), 0.1)
    with pytest.raises(RuntimeError, match=r"wan_cross_attn failed \(code 2\).*softmax_scale"):
        o.cross_attn(x, x, x, None, -0.1)
    assert o.rms_norm(x[:, :0], g, 1e-6).shape == (2, 0, 2, D)
    each = torch.vmap(lambda a: o.rms_norm(a, g, 1e-6))(torch.stack([x, 2 * x]))
    assert torch.equal(each[0], o.rms_norm(x, g, 1e-6)) and each.shape == (2, *x.shape)


def test_linear_is_torchs_where_the_kernel_does_not_take_it(W):
    """Other devices, types, layouts and sizes: torch's bits."""
    F = torch.nn.functional
    for x, w, b in ((torch.randn(2, 3, 64), torch.randn(256, 64), torch.randn(256)),
                    (torch.randn(2, 3, 65).bfloat16(), torch.randn(7, 65).bfloat16(), torch.randn(7).bfloat16()),
                    (torch.randn(5, 64).bfloat16(), torch.randn(256, 64).bfloat16(), torch.randn(256).bfloat16()),
                    (torch.randn(2, 0, 64), torch.randn(256, 64), torch.randn(256))):
        assert torch.equal(W.ops.linear(x, w, b), F.linear(x, w, b))


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["weight", "bias", "x"])
def test_linear_misaligned_is_torchs(W, which):
    """2560 and 2561 values from the start of an allocation: the address decides, and every operand that
    F.linear takes is taken."""
    t = {n: torch.randn(*s, device="cuda").bfloat16() for n, s in (("x", (2, 5, 64)), ("weight", (256, 64)), ("bias", (256,)))}
    flat = torch.zeros(t[which].numel() + 2561, device="cuda", dtype=torch.bfloat16)
    for off in (2560, 2561):
        view = flat[off:off + t[which].numel()].view(t[which].shape)
        view.copy_(t[which])
        args = {**t, which: view}
        got, want = W.ops.linear(**args).double(), args["x"].double() @ args["weight"].double().t() + args["bias"].double()
        assert ((got - want).abs() <= want.abs() * 2 ** -8 + 1e-3).all()
        if off % 8:
            assert torch.equal(W.ops.linear(**args), torch.nn.functional.linear(**{"input": args["x"], "weight": args["weight"],
                                                                                     "bias": args["bias"]}))


def _fresh(code, tmp_path):
    """Runs code in a new process over a copy of the package's Python files in tmp_path."""
    import shutil
    for f in os.listdir(__graft_entry__.PKG_DIR):
        if f.endswith(".py") or f == "libwan_attn.so":
            shutil.copy(os.path.join(__graft_entry__.PKG_DIR, f), tmp_path)
    code = (f"import sys, warnings, torch; sys.path.insert(0, {__graft_entry__.ROOT!r})\n"
            f"import __graft_entry__ as g; g.PKG_DIR = {str(tmp_path)!r}\n" + code)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    return r.stdout


def test_import_with_operators_that_do_not_load(tmp_path):
    """The package imports and its torch side runs; the first kernel call says what is wrong."""
    (tmp_path / f"libwan_ops-torch{torch.__version__}.so").write_bytes(b"not a library")
    (tmp_path / "libwan_ops.so").write_bytes(b"not a library")
    out = _fresh("""W = g.load_package()
m = W.model.random_model(W.model.WanConfig(dim=256, ffn_dim=512, num_heads=2, num_layers=1, in_dim=4, out_dim=4,
                                           text_dim=64, freq_dim=32), device="cpu", std=0.05)
fast = W.fast_dit.FastWanDiT(m, (1, 2, 2), 5.0, "sdpa", "sdpa", "eager")
fast.set_context(torch.zeros(1, 3, 64), torch.zeros(1, 3, 64))
print(tuple(fast(torch.zeros(4, 1, 4, 4), 1).shape))
try:
    W._native.lib()
except RuntimeError as e:
    print("does not load" in str(e))
""", tmp_path)
    assert out.split("\n")[:2] == ["(4, 1, 4, 4)", "True"]


def test_import_with_another_torch(tmp_path):
    """With operators built for another torch, which are not loaded, the Python functions are there, with
    a warning; with none built at all the first kernel call raises."""
    (tmp_path / "libwan_ops-torch0.1.so").write_bytes(b"not for this torch")
    out = _fresh("""W = g.load_package()
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    print(W._native.lib().wan_attn_abi_version(), len([w for w in seen if "another torch" in str(w.message)]))
""", tmp_path)
    assert out.split() == ["1", "1"]
    (tmp_path / "libwan_ops-torch0.1.so").unlink()
    out = _fresh("""W = g.load_package()
try:
    W._native.lib()
except RuntimeError as e:
    print("not built" in str(e))
""", tmp_path)
    assert out.split() == ["True"]
