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
    # split-K in half and in whole tiles; whole tiles, the last round whole or in halves; one round
    # of half tiles with weight-prefetch workgroups beside it
    (300, 1001, 10016, ("split", 10, 16, 2)), (512, 3073, 13824, ("split", 4, 56, 2)),
    (130, 17001, 6432, ("split", 3, 36, 4)), (4400, 5541, 96, ("tiles", 396, 0, 0)),
    (4352, 4099, 160, ("tiles", 256, 33, 0)), (700, 9003, 224, ("tiles", 0, 108, 40)),
]


@pytest.mark.parametrize("m,n,k,want", MX)
def test_mxfp8_and_fp8(m, n, k, want, hip):
    assert route("mx", m, n, k) == want
    x, w, bias = _inputs(m, n, k)
    qx, sx = ck.quantize_mxfp8(x)
    qw, sw = ck.quantize_mxfp8(w)
    product = ck.dequantize_mxfp8(qx, sx, torch.float32) @ ck.dequantize_mxfp8(qw, sw, torch.float32).t()
    _check(lambda b, o: ck.scaled_mm_mxfp8(qx, qw, sx, sw, bias=b, out_dtype=o), product, bias, m, n)
    # (codes of about 150 in the root mean square: sums of about 150^2 sqrt(K) = 2.6e6 at K = 13824, and
    # six times that, times 7.8e-4, is 1.2e4, inside f16's 65504)
    ta, tb = torch.full((1,), 0.37, device="cuda"), torch.full((1,), 0.0021, device="cuda")
    product = (qx.float() @ qw.float().t()) * (ta * tb)
    _check(lambda b, o: ck.scaled_mm_fp8(qx, qw, ta, tb, bias=b, out_dtype=o), product, bias, m, n)


NV = [  # 33-64 rows with two weight tiles per workgroup: short ragged K, long K, N past one round of small tiles
    (50, 9233, 928, ("skinny", 4, 2, 2, 0, 0)), (33, 8193, 96, ("skinny", 4, 2, 2, 0, 0)),
    (64, 8205, 8224, ("skinny", 4, 2, 2, 0, 0)), (40, 32771, 544, ("skinny", 4, 2, 2, 0, 0)),
    # the same with 1, 5, 9 and 10 chunks of 256 elements: its 4 waves hold 0 to 3 each
    (64, 32800, 224, ("skinny", 4, 2, 2, 0, 0)), (48, 32800, 1280, ("skinny", 4, 2, 2, 0, 0)),
    (64, 32801, 2304, ("skinny", 4, 2, 2, 0, 0)), (64, 32800, 2336, ("skinny", 4, 2, 2, 0, 0)),
    # split-K in half and in whole tiles; tiles as for MXFP8
    (300, 1001, 10016, ("split", 10, 4, 2)), (130, 17001, 6432, ("split", 3, 9, 4)),
    (4400, 5541, 96, ("tiles", 396, 0, 0)), (4352, 4099, 160, ("tiles", 256, 33, 0)),
    (700, 9003, 224, ("tiles", 0, 108, 0)),
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
