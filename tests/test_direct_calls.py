"""Calls that skip the custom op: the registry's shortcut accepts exactly what the general
validation accepts, and `direct` stands aside for everything that looks at or transforms an op."""
import itertools
import subprocess
import sys
from pathlib import Path

import pytest
import torch

import comfy_kitchen as ck
import comfy_kitchen.backends.hip as hb
from comfy_kitchen.constraints import FunctionConstraints, MinDims, ParamConstraint, validate_function_call
from comfy_kitchen.ops import direct, untouched
from comfy_kitchen.registry import BackendRegistry

PACKAGE = Path(__file__).resolve().parent.parent / "comfy-kitchen_amd"
ARCH = "gfx950:sramecc+:xnack-"
TABLE = hb._build_constraints()
DTYPES = [torch.float32, torch.bfloat16, torch.float16, torch.uint8, torch.int32, torch.float8_e4m3fn,
          torch.float8_e5m2, torch.float8_e8m0fnu]
SHAPES = [(), (1,), (4, 32), (3, 33), (2, 3, 4, 8), (0, 32), (1, 1, 2, 4, 2, 2)]


def _registry(arch):
    r = BackendRegistry()
    r._identity = ((9, 5), arch)
    return r


def _values():
    tensors = [torch.empty(s, dtype=d, device=dev) for s in SHAPES for d in DTYPES for dev in ("cpu", "meta")]
    return [None, *tensors, *DTYPES, 1.0, 3, "x"]


@pytest.mark.parametrize("arch", [ARCH, "gfx942", None])
@pytest.mark.parametrize("func", sorted(TABLE))
def test_shortcut_agrees_with_validation(func, arch):
    """Each parameter over every dtype, rank, divisibility and device (alone), each function with
    its devices as declared and widened to any."""
    reg = _registry(arch)
    rules = TABLE[func]
    anywhere = FunctionConstraints(
        params={n: ParamConstraint(p.dtypes, frozenset({"*"}), p.shape_rules) for n, p in rules.params.items()},
        default_devices=frozenset({"*"}), required_arch=rules.required_arch)
    accepted = 0
    for r in (rules, anywhere):
        for name, value in itertools.product(r.params, _values()):
            want = validate_function_call(r, {name: value}, compute_capability=(9, 5), arch=arch).success
            assert reg._accepts(r, {name: value}) == want, (func, name, value)
            accepted += want
    assert accepted > 0 or arch != ARCH


def test_shortcut_leaves_what_it_does_not_decide():
    class Odd(ParamConstraint):
        def check_dtype(self, value):
            return False

    reg = _registry(ARCH)
    x = torch.zeros(2, 2)
    assert reg._accepts(None, {"x": x})
    assert not reg._accepts(FunctionConstraints(params={"x": Odd()}), {"x": x})
    assert not reg._accepts(FunctionConstraints(min_compute_capability=(8, 0)), {"x": x})
    assert not reg._accepts(FunctionConstraints(params={"x": ParamConstraint(shape_rules=(MinDims(3),))}), {"x": x})


def test_cpu_and_odd_arguments_take_the_custom_op():
    x = torch.zeros(4, 32)
    assert not direct(x) and not direct(1.0) and not direct(None)
    with pytest.raises(Exception):
        ck.quantize_mxfp8(x)


@pytest.mark.gpu
def test_direct_conditions(hip):
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x = torch.randn(64, 128, device="cuda").bfloat16()
    assert direct(x) and direct(x, None, torch.nn.Parameter(x, requires_grad=False)) and direct(x, x.cpu())
    grad = x.clone().requires_grad_()
    assert not direct(grad) and not direct(x, grad)
    with torch.no_grad():
        assert direct(grad)
    assert not direct(x.cpu()) and not direct(x, 1.0)
    with Mode():
        assert not direct(x)
    with FakeTensorMode() as m:
        assert not direct(m.from_tensor(x))
    with torch.autograd.forward_ad.dual_level():
        assert not direct(x)
    with torch.autograd.profiler.profile():
        assert not direct(x)
    seen = []
    torch.vmap(lambda v: (seen.append(direct(x)), v)[1])(x)
    torch.jit.trace(lambda v: (seen.append(direct(v)), v + 1)[1], (x,), check_trace=False)
    assert seen and not any(seen)


@pytest.mark.gpu
def test_direct_equals_custom_op(hip):
    """The same results by either way, on another stream too, and a gradient is refused as before."""
    x = torch.randn(70, 160, device="cuda").bfloat16()
    op = torch.ops.comfy_kitchen
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        q, s = ck.quantize_mxfp8(x, pad_32x=True)
    torch.cuda.current_stream().wait_stream(side)
    oq, os = op.quantize_mxfp8(x, True)
    assert torch.equal(q.view(torch.uint8), oq.view(torch.uint8)) and torch.equal(s.view(torch.uint8), os.view(torch.uint8))
    assert q.dtype == oq.dtype and s.dtype == os.dtype and s.shape == os.shape
    assert torch.equal(ck.scaled_mm_mxfp8(q, q, s, s), op.scaled_mm_mxfp8(q, q, s, s, None, 2))
    for tensors in (ck.quantize_nvfp4_dynamic(x), ck.quantize_fp8_dynamic(x)):
        assert all(type(t) is torch.Tensor and not t.requires_grad for t in tensors)
    y = ck.dequantize_per_tensor_fp8(ck.quantize_per_tensor_fp8(x.clone().requires_grad_(), torch.ones(1, device="cuda")),
                                     torch.ones(1, device="cuda"))
    with pytest.raises(RuntimeError):
        y.float().sum().backward()


@pytest.mark.gpu
def test_lazy_views_take_the_custom_op(hip):
    """A negated view's memory holds the values before the negation: as input, as scale (a complex
    number's conjugated imaginary part is one) and as bias it gives what a plain copy gives."""
    x = torch.randn(64, 128, device="cuda").bfloat16()
    neg, z = torch._neg_view(x), torch.conj(torch.tensor([[1.5 - 0.25j]], device="cuda"))
    scale = z.imag.reshape(1)
    assert neg.is_neg() and scale.is_neg()
    zeros = torch._efficientzerotensor((4, 128), dtype=torch.bfloat16, device="cuda")
    assert not direct(neg) and not direct(x, scale) and not direct(zeros)
    for a, b in zip(ck.quantize_mxfp8(neg), ck.quantize_mxfp8(-x)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    plain = torch.full((1,), 0.25, device="cuda")
    assert torch.equal(plain, scale)
    got, want = ck.quantize_per_tensor_fp8(x, scale), ck.quantize_per_tensor_fp8(x, plain)
    assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    q, s = ck.quantize_mxfp8(x)
    bias = torch.randn(64, device="cuda")
    assert torch.equal(ck.scaled_mm_mxfp8(q, q, s, s, bias=torch._neg_view(bias)), ck.scaled_mm_mxfp8(q, q, s, s, bias=-bias))
    assert ck.quantize_mxfp8(zeros)[0].float().abs().sum() == 0


OPS = ["amax_scale", "apply_rope", "apply_rope1", "dequantize_fp8", "dequantize_mxfp8", "dequantize_nvfp4",
       "quantize_fp8", "quantize_fp8_dynamic", "quantize_mxfp8", "quantize_nvfp4", "quantize_nvfp4_dynamic",
       "scaled_mm_fp8", "scaled_mm_mxfp8", "scaled_mm_nvfp4"]


@pytest.mark.parametrize("op", OPS)
def test_registered_kernels_are_seen(op):
    """A kernel that a program puts on one of the ops, at any key a plain GPU tensor would meet,
    ends the shortcut for that op, until the program takes it back."""
    assert untouched(op)
    for key in ("CUDA", "AutocastCUDA", "AutogradCUDA", "ADInplaceOrView"):
        lib = torch.library.Library("comfy_kitchen", "IMPL")
        lib.impl(op, lambda *args: None, key)
        assert not untouched(op), key
        lib._destroy()
        assert untouched(op)


def test_custom_op_registrations_are_seen():
    """register_kernel and register_autocast last as long as the process, so in one of its own."""
    code = f"""
import sys
sys.path.insert(0, {str(PACKAGE)!r})
import torch
import comfy_kitchen.ops as ops
assert ops.untouched("quantize_fp8") and ops.untouched("quantize_mxfp8") and ops.untouched("apply_rope1")
ops.quantize_fp8.register_kernel("cuda")(lambda x, scale, code: x)
torch.library.register_kernel("comfy_kitchen::apply_rope1", "cuda", lambda x, f: x)
ops.quantize_mxfp8.register_autocast("cuda", torch.float32)
assert not ops.untouched("quantize_fp8") and not ops.untouched("quantize_mxfp8") and not ops.untouched("apply_rope1")
print("ok")
"""
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert run.stdout.strip() == "ok", run.stderr


@pytest.mark.gpu
def test_registered_kernel_serves_the_call(hip):
    x, scale = torch.randn(4, 32, device="cuda").bfloat16(), torch.ones(1, device="cuda")
    marker = torch.zeros(4, 32, device="cuda")
    lib = torch.library.Library("comfy_kitchen", "IMPL")
    lib.impl("quantize_fp8", lambda x, scale, code: marker, "CUDA")
    lib.impl("quantize_mxfp8", lambda x, pad: (marker, marker), "AutocastCUDA")
    try:
        assert torch.equal(ck.quantize_per_tensor_fp8(x, scale), marker)
        assert ck.quantize_mxfp8(x)[0].dtype == torch.float8_e4m3fn  # no autocast here: the rule sleeps
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert ck.quantize_mxfp8(x)[0].dtype == torch.float32
    finally:
        lib._destroy()
    assert ck.quantize_per_tensor_fp8(x, scale).dtype == torch.float8_e4m3fn


@pytest.mark.parametrize("holder,name", [("torch._C._functorch", "peek_interpreter_stack"),
                                         ("torch._C._autograd", "_profiler_enabled"),
                                         ("torch._C", "_get_tracing_state"),
                                         ("torch.autograd.forward_ad", "_current_level")])
def test_torch_without_a_probe_takes_the_custom_op(holder, name):
    """Where torch lacks one of the names the shortcut asks, the package imports and every call
    takes the custom op (here: reaches the registry, which has no backend for a CPU tensor)."""
    code = f"""
import sys
sys.path.insert(0, {str(PACKAGE)!r})
import torch, torch.autograd.forward_ad
del {holder}.{name}
import comfy_kitchen as ck
from comfy_kitchen.ops import direct
x = torch.zeros(4, 32)
assert not direct(x)
try:
    ck.quantize_mxfp8(x)
except ck.NoCapableBackendError:
    print("ok")
"""
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert run.stdout.strip() == "ok", run.stderr


@pytest.mark.gpu
def test_no_probes_same_results(hip, monkeypatch):
    import comfy_kitchen.ops as ops

    x = torch.randn(16, 64, device="cuda").bfloat16()
    want = ck.quantize_mxfp8(x)
    monkeypatch.setattr(ops, "_OBSERVABLE", False)
    assert not direct(x)
    got = ck.quantize_mxfp8(x)
    assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, want))
