"""torch.library custom ops `comfy_kitchen::*` and their fake (meta) implementations.

Op names, argument order, dtype codes and output shapes follow the reference
(backends/eager/quantization.py:31-39 for the codes, 411-730 for the quantization
ops, backends/eager/rope.py:26-58 for RoPE).  Each op body asks the registry for a
backend implementation and calls it with the eager backend's keyword arguments; the
fake implementations give torch.compile the output shapes without running anything.
"""
from __future__ import annotations

import torch
import torch.autograd.forward_ad as _forward_ad

from .float_utils import roundup
from .registry import registry

DTYPE_CODE_TO_DTYPE = {
    0: torch.float32,
    1: torch.float16,
    2: torch.bfloat16,
    5: torch.float8_e4m3fn,
    6: torch.float8_e5m2,
}
DTYPE_TO_CODE = {v: k for k, v in DTYPE_CODE_TO_DTYPE.items()}


def _dispatch(func_name: str, **kwargs):
    return registry.get_implementation(func_name, kwargs=kwargs)(**kwargs)


_Tensor, _Parameter = torch.Tensor, torch.nn.Parameter
_C = torch._C
try:
    _is_compiling = torch.compiler.is_compiling
    _dispatch_modes, _function_modes = _C._len_torch_dispatch_stack, _C._len_torch_function_stack
    _transforms, _tracing = _C._functorch.peek_interpreter_stack, _C._get_tracing_state
    _profiling = _C._autograd._profiler_enabled
    torch.Tensor._is_zerotensor
    _forward_ad._current_level
    _registered = torch.library._impls  # "namespace/op/key" of every kernel registered from Python
    _registered.isdisjoint
    _OBSERVABLE = True
except AttributeError:
    # A torch that lacks one of these (several are not public) gives no way to tell whether
    # something looks at the op: every call takes the custom op then.
    _OBSERVABLE = False

# Every key at which the dispatcher could find a kernel for plain GPU tensors ahead of, or in place
# of, the custom op's own (which it holds under alias keys, so none of these is set by it).
_KERNEL_KEYS = ("CUDA", "AutocastCUDA", "AutogradCUDA", "ADInplaceOrView")


class _Kernels(dict):
    """op name -> the entries that a program's own kernels for it make in torch's list."""

    def __missing__(self, op: str) -> frozenset:
        entries = self[op] = frozenset(f"comfy_kitchen/{op}/{key}" for key in _KERNEL_KEYS)
        return entries


_kernels = _Kernels()


def untouched(op: str) -> bool:
    """Whether no program has registered a kernel of its own (torch.library, an autocast rule,
    the custom op's register_kernel) for GPU tensors on `comfy_kitchen::<op>`: one that has
    expects `ck.*` calls to reach it.  (Not seen: a kernel registered in C++, and one put in
    place of the op's default under the default's own alias key.)  About 0.15 us a call; asking
    the dispatcher itself took 0.7."""
    return _registered.isdisjoint(_kernels[op])


def direct(*tensors) -> bool:
    """Whether a `ck.*` call may go to the registry without the custom op around it: nothing
    looks at or transforms the op (compilation and tracing, dispatch and function modes, vmap
    and the other function transforms, forward-mode AD, the profiler), the first tensor is on
    the GPU, and every tensor is a plain one that no gradient is asked of and whose memory holds
    its values (a lazily negated view's does not, and a zero tensor has none: the dispatcher makes
    them plain before the custom op's kernel sees them; complex tensors, which alone can be lazily
    conjugated, no backend function takes).  Anything else takes
    the custom op, which serves all of these.  The custom op's Python layers cost more than the
    call itself: on a 77 x 4096 tensor quantize_per_tensor_fp8 and dequantize_per_tensor_fp8
    took 20 us each from Python for 2.7 us on the GPU."""
    if (not _OBSERVABLE or _is_compiling() or _dispatch_modes() or _function_modes() or _transforms() is not None
            or _tracing() is not None or _profiling() or _forward_ad._current_level >= 0):
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        kind = type(t)
        if kind is _Tensor or kind is _Parameter:
            if grad and t.requires_grad or t.is_neg() or t._is_zerotensor():
                return False
        elif t is not None:
            return False
    first = tensors[0]
    return first is not None and first.is_cuda


# --------------------------------------------------------------- per-tensor FP8
@torch.library.custom_op("comfy_kitchen::quantize_fp8", mutates_args=())
def quantize_fp8(x: torch.Tensor, scale: torch.Tensor, output_dtype_code: int) -> torch.Tensor:
    return _dispatch("quantize_per_tensor_fp8", x=x, scale=scale,
                     output_type=DTYPE_CODE_TO_DTYPE[output_dtype_code])


@quantize_fp8.register_fake
def _(x, scale, output_dtype_code):
    return torch.empty_like(x, dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code])


@torch.library.custom_op("comfy_kitchen::dequantize_fp8", mutates_args=())
def dequantize_fp8(x: torch.Tensor, scale: torch.Tensor, output_dtype_code: int) -> torch.Tensor:
    return _dispatch("dequantize_per_tensor_fp8", x=x, scale=scale,
                     output_type=DTYPE_CODE_TO_DTYPE[output_dtype_code])


@dequantize_fp8.register_fake
def _(x, scale, output_dtype_code):
    return torch.empty_like(x, dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code])


def _quantize_fp8_dynamic(x: torch.Tensor, divisor: float, output_type: torch.dtype) -> tuple[torch.Tensor, torch.Tensor]:
    """The fused call where one backend serves it and the quantizer; else the two calls it stands
    for, each from the backend that the program has chosen for it."""
    fused = registry.shared_implementation("quantize_fp8_dynamic", "quantize_per_tensor_fp8",
                                           {"x": x, "output_type": output_type})
    if fused is not None:
        return fused(x=x, divisor=divisor, output_type=output_type)
    scale = _dispatch("amax_scale", x=x, divisor=divisor)
    return _dispatch("quantize_per_tensor_fp8", x=x, scale=scale, output_type=output_type), scale


@torch.library.custom_op("comfy_kitchen::quantize_fp8_dynamic", mutates_args=())
def quantize_fp8_dynamic(x: torch.Tensor, divisor: float, output_dtype_code: int) -> tuple[torch.Tensor, torch.Tensor]:
    return _quantize_fp8_dynamic(x, divisor, DTYPE_CODE_TO_DTYPE[output_dtype_code])


@quantize_fp8_dynamic.register_fake
def _(x, divisor, output_dtype_code):
    return (torch.empty_like(x, dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code]),
            torch.empty((), dtype=torch.float32, device=x.device))


# ------------------------------------------------------------------------ NVFP4
@torch.library.custom_op("comfy_kitchen::quantize_nvfp4", mutates_args=())
def quantize_nvfp4(x: torch.Tensor, per_tensor_scale: torch.Tensor, epsilon: float,
                   pad_16x: bool, hi_first: bool) -> tuple[torch.Tensor, torch.Tensor]:
    return _dispatch("quantize_nvfp4", x=x, per_tensor_scale=per_tensor_scale,
                     epsilon=epsilon, pad_16x=pad_16x, hi_first=hi_first)


@quantize_nvfp4.register_fake
def _(x, per_tensor_scale, epsilon, pad_16x, hi_first):
    rows, cols = x.shape
    if pad_16x:
        rows, cols = roundup(rows, 16), roundup(cols, 16)
    q = torch.empty((rows, cols // 2), dtype=torch.uint8, device=x.device)
    s = torch.empty((roundup(rows, 128), roundup(cols // 16, 4)), dtype=torch.float8_e4m3fn, device=x.device)
    return q, s


@torch.library.custom_op("comfy_kitchen::quantize_nvfp4_dynamic", mutates_args=())
def quantize_nvfp4_dynamic(x: torch.Tensor, divisor: float, pad_16x: bool,
                           hi_first: bool) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    return _dispatch("quantize_nvfp4_dynamic", x=x, divisor=divisor, pad_16x=pad_16x, hi_first=hi_first)


@quantize_nvfp4_dynamic.register_fake
def _(x, divisor, pad_16x, hi_first):
    rows, cols = x.shape
    if pad_16x:
        rows, cols = roundup(rows, 16), roundup(cols, 16)
    q = torch.empty((rows, cols // 2), dtype=torch.uint8, device=x.device)
    s = torch.empty((roundup(rows, 128), roundup(cols // 16, 4)), dtype=torch.float8_e4m3fn, device=x.device)
    return q, s, torch.empty((), dtype=torch.float32, device=x.device)


@torch.library.custom_op("comfy_kitchen::dequantize_nvfp4", mutates_args=())
def dequantize_nvfp4(qx: torch.Tensor, per_tensor_scale: torch.Tensor, block_scales: torch.Tensor,
                     output_dtype_code: int, hi_first: bool) -> torch.Tensor:
    return _dispatch("dequantize_nvfp4", qx=qx, per_tensor_scale=per_tensor_scale,
                     block_scales=block_scales, output_type=DTYPE_CODE_TO_DTYPE[output_dtype_code],
                     hi_first=hi_first)


@dequantize_nvfp4.register_fake
def _(qx, per_tensor_scale, block_scales, output_dtype_code, hi_first):
    rows, cols = qx.shape
    return torch.empty((rows, cols * 2), dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code], device=qx.device)


@torch.library.custom_op("comfy_kitchen::scaled_mm_nvfp4", mutates_args=())
def scaled_mm_nvfp4(a: torch.Tensor, b: torch.Tensor, tensor_scale_a: torch.Tensor,
                    tensor_scale_b: torch.Tensor, block_scale_a: torch.Tensor,
                    block_scale_b: torch.Tensor, bias: torch.Tensor | None,
                    output_dtype_code: int, alpha: torch.Tensor | None) -> torch.Tensor:
    return _dispatch("scaled_mm_nvfp4", a=a, b=b, tensor_scale_a=tensor_scale_a,
                     tensor_scale_b=tensor_scale_b, block_scale_a=block_scale_a,
                     block_scale_b=block_scale_b, bias=bias,
                     out_dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code], alpha=alpha)


@scaled_mm_nvfp4.register_fake
def _(a, b, tensor_scale_a, tensor_scale_b, block_scale_a, block_scale_b, bias, output_dtype_code, alpha):
    return torch.empty((a.shape[0], b.shape[0]), dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code], device=a.device)


# ------------------------------------------------------------- dynamic scales
@torch.library.custom_op("comfy_kitchen::amax_scale", mutates_args=())
def amax_scale(x: torch.Tensor, divisor: float) -> torch.Tensor:
    return _dispatch("amax_scale", x=x, divisor=divisor)


@amax_scale.register_fake
def _(x, divisor):
    return torch.empty((), dtype=torch.float32, device=x.device)


# ------------------------------------------------------------------------ MXFP8
@torch.library.custom_op("comfy_kitchen::quantize_mxfp8", mutates_args=())
def quantize_mxfp8(x: torch.Tensor, pad_32x: bool) -> tuple[torch.Tensor, torch.Tensor]:
    return _dispatch("quantize_mxfp8", x=x, pad_32x=pad_32x)


@quantize_mxfp8.register_fake
def _(x, pad_32x):
    rows, cols = x.shape
    if pad_32x:
        rows, cols = roundup(rows, 32), roundup(cols, 32)
    q = torch.empty((rows, cols), dtype=torch.float8_e4m3fn, device=x.device)
    s = torch.empty((roundup(rows, 128), roundup(cols // 32, 4)), dtype=torch.float8_e8m0fnu, device=x.device)
    return q, s


@torch.library.custom_op("comfy_kitchen::dequantize_mxfp8", mutates_args=())
def dequantize_mxfp8(qx: torch.Tensor, block_scales: torch.Tensor, output_dtype_code: int) -> torch.Tensor:
    return _dispatch("dequantize_mxfp8", qx=qx, block_scales=block_scales,
                     output_type=DTYPE_CODE_TO_DTYPE[output_dtype_code])


@dequantize_mxfp8.register_fake
def _(qx, block_scales, output_dtype_code):
    return torch.empty_like(qx, dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code])


@torch.library.custom_op("comfy_kitchen::scaled_mm_mxfp8", mutates_args=())
def scaled_mm_mxfp8(a: torch.Tensor, b: torch.Tensor, block_scale_a: torch.Tensor,
                    block_scale_b: torch.Tensor, bias: torch.Tensor | None,
                    output_dtype_code: int) -> torch.Tensor:
    return _dispatch("scaled_mm_mxfp8", a=a, b=b, block_scale_a=block_scale_a,
                     block_scale_b=block_scale_b, bias=bias,
                     out_dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code])


@scaled_mm_mxfp8.register_fake
def _(a, b, block_scale_a, block_scale_b, bias, output_dtype_code):
    return torch.empty((a.shape[0], b.shape[0]), dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code], device=a.device)


@torch.library.custom_op("comfy_kitchen::scaled_mm_fp8", mutates_args=())
def scaled_mm_fp8(a: torch.Tensor, b: torch.Tensor, scale_a: torch.Tensor, scale_b: torch.Tensor,
                  bias: torch.Tensor | None, output_dtype_code: int) -> torch.Tensor:
    return _dispatch("scaled_mm_fp8", a=a, b=b, scale_a=scale_a, scale_b=scale_b, bias=bias,
                     out_dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code])


@scaled_mm_fp8.register_fake
def _(a, b, scale_a, scale_b, bias, output_dtype_code):
    return torch.empty((a.shape[0], b.shape[0]), dtype=DTYPE_CODE_TO_DTYPE[output_dtype_code], device=a.device)


# ------------------------------------------------------------------------- RoPE
@torch.library.custom_op("comfy_kitchen::apply_rope", mutates_args=())
def apply_rope(xq: torch.Tensor, xk: torch.Tensor, freqs_cis: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    return _dispatch("apply_rope", xq=xq, xk=xk, freqs_cis=freqs_cis)


@apply_rope.register_fake
def _(xq, xk, freqs_cis):
    return torch.empty_like(xq), torch.empty_like(xk)


@torch.library.custom_op("comfy_kitchen::apply_rope1", mutates_args=())
def apply_rope1(x: torch.Tensor, freqs_cis: torch.Tensor) -> torch.Tensor:
    return _dispatch("apply_rope1", x=x, freqs_cis=freqs_cis)


@apply_rope1.register_fake
def _(x, freqs_cis):
    return torch.empty_like(x)
