"""Every kernel that a GEMM call can select, by sizes that select it (asserted), against an fp32
matmul of the dequantized operands: rows past M, columns past N (N odd, so that elements are
stored one by one, or a multiple of 8), K ending inside a stage, with and without a bias, in
every output type."""
import pytest
import torch

import comfy_kitchen as ck
from routes import route

pytestmark = pytest.mark.gpu

# fp32 output: the order of the fp32 sums; 16-bit outputs: one rounding (2^-9 and 2^-12 relative)
REL = {torch.float32: 1e-4, torch.float16: 1e-3, torch.bfloat16: 4e-3}
OUTPUTS = [(torch.float32, None), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
           (torch.bfloat16, None), (torch.float32, torch.float16)]


def _rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


def _inputs(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda") * torch.exp(torch.randn(m, 1, generator=g, device="cuda"))
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    return x.bfloat16(), w.bfloat16(), torch.randn(n, generator=g, device="cuda")


def _check(call, product, bias, m, n):
    for out_dtype, bias_dtype in OUTPUTS:
        b = None if bias_dtype is None else bias.to(bias_dtype)
        got = call(b, out_dtype)
        assert got.shape == (m, n) and got.dtype == out_dtype
        rel = _rel(got, product if b is None else product + b.float())
        assert rel <= REL[out_dtype], (out_dtype, bias_dtype, rel)
    return call(None, torch.float32)


MX = [  # 17-64 rows: the skinny forms that the small tiles leave
    (25, 8205, 1056, ("skinny", 4, 2, 1, 32, 0)), (18, 16401, 544, ("skinny", 2, 1, 1, 32, 0)),
    (29, 20401, 4128, ("skinny", 4, 1, 1, 32, 0)), (32, 24579, 96, ("skinny", 2, 2, 1, 32, 0)),
    (52, 16403, 544, ("skinny", 2, 1, 2, 64, 0)), (33, 24576, 1216, ("skinny", 2, 1, 2, 64, 0)),
    (64, 32771, 160, ("skinny", 2, 2, 2, 64, 0)), (40, 33001, 672, ("skinny", 2, 2, 2, 64, 0)),
]


@pytest.mark.parametrize("m,n,k,want", MX)
def test_mxfp8_and_fp8(m, n, k, want, hip):
    assert route("mx", m, n, k) == want
    x, w, bias = _inputs(m, n, k)
    qx, sx = ck.quantize_mxfp8(x)
    qw, sw = ck.quantize_mxfp8(w)
    product = ck.dequantize_mxfp8(qx, sx, torch.float32) @ ck.dequantize_mxfp8(qw, sw, torch.float32).t()
    _check(lambda b, o: ck.scaled_mm_mxfp8(qx, qw, sx, sw, bias=b, out_dtype=o), product, bias, m, n)
    ta, tb = torch.full((1,), 0.37, device="cuda"), torch.full((1,), 0.021, device="cuda")
    product = (qx.float() @ qw.float().t()) * (ta * tb)
    _check(lambda b, o: ck.scaled_mm_fp8(qx, qw, ta, tb, bias=b, out_dtype=o), product, bias, m, n)


NV = [  # 33-64 rows with two weight tiles per workgroup: short ragged K, long K, N past one round of small tiles
    (50, 9233, 928, ("skinny", 4, 2, 2, 0, 0)), (33, 8193, 96, ("skinny", 4, 2, 2, 0, 0)),
    (64, 8205, 8224, ("skinny", 4, 2, 2, 0, 0)), (40, 32771, 544, ("skinny", 4, 2, 2, 0, 0)),
]


@pytest.mark.parametrize("m,n,k,want", NV)
def test_nvfp4(m, n, k, want, hip):
    assert route("nv", m, n, k) == want
    x, w, bias = _inputs(m, n, k)
    qx, sx, gx = ck.quantize_nvfp4_dynamic(x)
    qw, sw, gw = ck.quantize_nvfp4_dynamic(w)
    product = ck.dequantize_nvfp4(qx, gx, sx, torch.float32) @ ck.dequantize_nvfp4(qw, gw, sw, torch.float32).t()
    scaled = _check(lambda b, o: ck.scaled_mm_nvfp4(qx, qw, gx, gw, sx, sw, bias=b, out_dtype=o), product, bias, m, n)
    # two tensor scales give the bits that their fp32 product, passed as alpha, gives
    alpha = ck.scaled_mm_nvfp4(qx, qw, gx, gw, sx, sw, alpha=gx * gw, out_dtype=torch.float32)
    assert torch.equal(scaled, alpha)
