"""The small-tile GEMMs of a few hundred activation rows, every tile shape: rows past M, columns
past N (N odd, so that elements are stored one by one, and N a multiple of 8), K ending inside
a stage, one to three stages (fewer than the ring holds), bias and output types, against an
fp32 matmul of the dequantized operands."""
import pytest
import torch

import comfy_kitchen as ck
from routes import route

pytestmark = pytest.mark.gpu

# fp32 output: the order of the fp32 sums; 16-bit outputs: one rounding (2^-9 and 2^-12 relative)
REL = {torch.float32: 1e-4, torch.float16: 1e-3, torch.bfloat16: 4e-3}

# (m, n, k, tile): one stage, three stages, many; at most 64 rows, then more
SHAPES = [(17, 10248, 3104, (64, 64)), (33, 8192, 96, (64, 64)), (64, 16384, 160, (64, 64)), (33, 17001, 1312, (64, 128)),
          (20, 32767, 4128, (64, 128)), (65, 33, 32, (64, 64)), (70, 1000, 352, (64, 64)), (200, 2001, 1152, (64, 64)),
          (200, 7001, 1056, (128, 64)), (201, 6992, 128, (128, 64)), (300, 7001, 1120, (128, 96)),
          (300, 9003, 2080, (128, 128)), (500, 9008, 2080, (128, 160)), (500, 9004, 2112, (128, 160)),
          (500, 11001, 4128, (128, 192)), (512, 12288, 4096, (128, 192))]


def _rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


@pytest.mark.parametrize("out_dtype,bias_dtype", [(torch.float32, None), (torch.bfloat16, torch.bfloat16),
                                                  (torch.float16, torch.float32), (torch.bfloat16, None)])
@pytest.mark.parametrize("m,n,k,tile", SHAPES)
def test_small_tiles(m, n, k, tile, out_dtype, bias_dtype, hip):
    assert route("mx", m, n, k) == ("small", *tile)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda") * torch.exp(torch.randn(m, 1, generator=g, device="cuda"))
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    bias = None if bias_dtype is None else torch.randn(n, generator=g, device="cuda").to(bias_dtype)
    b32 = 0.0 if bias is None else bias.float()
    qx, sx = ck.quantize_mxfp8(x.bfloat16())
    qw, sw = ck.quantize_mxfp8(w.bfloat16())
    want = ck.dequantize_mxfp8(qx, sx, torch.float32) @ ck.dequantize_mxfp8(qw, sw, torch.float32).t() + b32
    got = ck.scaled_mm_mxfp8(qx, qw, sx, sw, bias=bias, out_dtype=out_dtype)
    assert got.shape == (m, n) and got.dtype == out_dtype
    assert _rel(got, want) <= REL[out_dtype]
    ta, tb = torch.full((1,), 0.37, device="cuda"), torch.full((1,), 0.021, device="cuda")
    want = (qx.float() @ qw.float().t()) * (ta * tb) + b32
    got = ck.scaled_mm_fp8(qx, qw, ta, tb, bias=bias, out_dtype=out_dtype)
    assert _rel(got, want) <= REL[out_dtype]


# (m, n, k, tile): part of a line, two lines, an odd number of them
NV_SHAPES = [(33, 8200, 1312, (64, 64)), (64, 17001, 1056, (64, 128)), (40, 8192, 256, (64, 64)), (65, 33, 32, (64, 64)),
             (70, 1000, 480, (64, 64)), (200, 2001, 1312, (64, 64)), (200, 7001, 1056, (64, 128)),
             (201, 6992, 256, (64, 128)), (300, 9003, 2080, (128, 128)), (500, 7000, 800, (128, 128)),
             (500, 9004, 2112, (128, 192)), (512, 12288, 1024, (128, 192))]


@pytest.mark.parametrize("out_dtype,bias_dtype", [(torch.float32, None), (torch.bfloat16, torch.bfloat16),
                                                  (torch.float16, torch.float32), (torch.bfloat16, None)])
@pytest.mark.parametrize("m,n,k,tile", NV_SHAPES)
def test_small_tiles_nvfp4(m, n, k, tile, out_dtype, bias_dtype, hip):
    assert route("nv", m, n, k) == ("small", *tile)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda") * torch.exp(torch.randn(m, 1, generator=g, device="cuda"))
    w = torch.randn(n, k, generator=g, device="cuda") * 0.02
    bias = None if bias_dtype is None else torch.randn(n, generator=g, device="cuda").to(bias_dtype)
    qx, sx, gx = ck.quantize_nvfp4_dynamic(x.bfloat16())
    qw, sw, gw = ck.quantize_nvfp4_dynamic(w.bfloat16())
    want = ck.dequantize_nvfp4(qx, gx, sx, torch.float32) @ ck.dequantize_nvfp4(qw, gw, sw, torch.float32).t()
    want = want + (0.0 if bias is None else bias.float())
    got = ck.scaled_mm_nvfp4(qx, qw, gx, gw, sx, sw, bias=bias, out_dtype=out_dtype)
    assert got.shape == (m, n) and got.dtype == out_dtype
    assert _rel(got, want) <= REL[out_dtype]


def test_small_tiles_read_no_neighbour(hip):
    """Operands inside larger buffers full of NaN codes: nothing outside them is used."""
    m, n, k = 129, 97, 160
    assert route("mx", m, n, k)[0] == "small"
    pad = torch.full((m + n + 8, k), 0x7F, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn)
    x, _ = ck.quantize_mxfp8(torch.randn(m, k, device="cuda").bfloat16())
    w, _ = ck.quantize_mxfp8(torch.randn(n, k, device="cuda").bfloat16())
    pad.view(torch.uint8)[:m] = x.view(torch.uint8)
    pad.view(torch.uint8)[m + 4:m + 4 + n] = w.view(torch.uint8)
    one = torch.ones(1, device="cuda")
    got = ck.scaled_mm_fp8(pad[:m], pad[m + 4:m + 4 + n], one, one, out_dtype=torch.float32)
    assert _rel(got, x.float() @ w.float().t()) <= 1e-4


@pytest.mark.parametrize("m,kinds", [(3, ("skinny", "skinny")), (40, ("skinny", "skinny")), (100, ("small", "split")),
                                     (4352, ("tiles", "split"))])
def test_nvfp4_tensor_scales_multiplied_in_the_kernel(m, kinds, hip):
    """Two tensor scales give the bits that their fp32 product, passed as alpha, gives: skinny,
    small-tile and whole-tile kernels, and split-K (its reduce kernel)."""
    for (n, k), kind in zip(((4000, 64), (1000, 8192)), kinds):
        assert route("nv", m, n, k)[0] == kind
        qx, sx, gx = ck.quantize_nvfp4_dynamic(torch.randn(m, k, device="cuda").bfloat16())
        qw, sw, gw = ck.quantize_nvfp4_dynamic(torch.randn(n, k, device="cuda").bfloat16())
        got = ck.scaled_mm_nvfp4(qx, qw, gx, gw, sx, sw, out_dtype=torch.float32)
        assert torch.equal(got, ck.scaled_mm_nvfp4(qx, qw, gx, gw, sx, sw, alpha=gx * gw, out_dtype=torch.float32))
