"""The dynamic-scale quantizers at the edges of their launch forms, and the 16-bit fast
paths of the block quantizers on inputs padded in rows: bit-exact against the separate
calls (amax_scale, then the quantizer) and the CPU oracle.

Edges: one launch up to 64 KB of input and two above, 1024 elements (the smallest for the
per-tensor kernel's fused form), element counts that are no multiple of 8, unaligned views,
and the sizes at which the reduction's grid changes (512 workgroups of 2 loads a thread)."""
import pytest
import torch

import comfy_kitchen as ck
from conftest import bits
from oracle import eager_ref as ref

pytestmark = pytest.mark.gpu

E4M3, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2
SPREAD = 512 * 256 * 2 * 8  # elements of 16 bits in 512 workgroups of 2 loads a thread


def _x(n, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(n + seed)
    return (3 * torch.randn(n, generator=g, device="cuda")).to(dtype)


@pytest.mark.parametrize("out", [E4M3, E5M2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1032, 5001, 32768 - 8, 32768, 32768 + 8, 32769, 98304, SPREAD - 8,
                               SPREAD + 8])
def test_fp8_dynamic(n, dtype, out, hip):
    x = _x(n, dtype)
    x[n // 2] = -7.5  # the largest magnitude need not be anywhere special
    x[n - 1] = 31.0
    limit = torch.finfo(out).max
    for v in (x, _x(n + 1, dtype)[1:]):  # aligned, and one element past alignment
        q, s = ck.quantize_fp8_dynamic(v, limit, out)
        want = ck.amax_scale(v, limit)
        assert s.shape == () and torch.equal(s, want)
        assert torch.equal(bits(q), bits(ck.quantize_per_tensor_fp8(v, want, out)))
        assert torch.equal(s.cpu(), ref.default_scale(v.cpu(), limit))


@pytest.mark.parametrize("case", ["nan", "inf", "zero"])
@pytest.mark.parametrize("n", [4096, 65536])
def test_fp8_dynamic_special(n, case, hip):
    x = _x(n, torch.bfloat16)
    if case == "zero":
        x.zero_()
    else:
        x[n - 3] = float(case)
    q, s = ck.quantize_fp8_dynamic(x)
    want = ck.amax_scale(x, 448.0)
    assert torch.equal(bits(s), bits(want))
    assert torch.equal(bits(q), bits(ck.quantize_per_tensor_fp8(x, want)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k", [(1, 64), (1, 3072), (4, 3072), (15, 1088), (17, 1984), (32, 1024), (33, 1024),
                                 (129, 256), (300, 3072)])
def test_nvfp4_rows_padded(m, k, dtype, hip):
    x = _x(m * k, dtype).reshape(m, k)
    q, s, g = ck.quantize_nvfp4_dynamic(x, 2688.0, pad_16x=True)
    want = ck.amax_scale(x, 2688.0)
    assert torch.equal(g, want)
    rq, rs = ref.quantize_nvfp4(x.cpu(), want.cpu(), pad_16x=True)
    assert torch.equal(q.cpu(), rq) and torch.equal(bits(s), bits(rs))
    q, s = ck.quantize_nvfp4(x, want, pad_16x=True)
    assert torch.equal(q.cpu(), rq) and torch.equal(bits(s), bits(rs))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k", [(1, 128), (1, 3072), (31, 256), (33, 1152), (130, 384), (1333, 3072)])
def test_mxfp8_rows_padded(m, k, dtype, hip):
    x = _x(m * k, dtype).reshape(m, k)
    q, s = ck.quantize_mxfp8(x, pad_32x=True)
    rq, rs = ref.quantize_mxfp8(x.cpu(), pad_32x=True)
    assert torch.equal(bits(q), bits(rq)) and torch.equal(bits(s), bits(rs))


@pytest.mark.parametrize("hi_first", [True, False])
@pytest.mark.parametrize("m", [1022, 1025])  # either side of the size from which the fast path serves them
def test_nvfp4_rows_padded_given_scale(m, hi_first, hip):
    x = _x(m * 3072, torch.bfloat16).reshape(m, 3072)
    g = ck.amax_scale(x, 2688.0)
    q, s = ck.quantize_nvfp4(x, g, pad_16x=True, hi_first=hi_first)
    rq, rs = ref.quantize_nvfp4(x.cpu(), g.cpu(), pad_16x=True, hi_first=hi_first)
    assert torch.equal(q.cpu(), rq) and torch.equal(bits(s), bits(rs))
