"""The tile GEMMs' bias: staged in LDS as fp32 and added to the fp32 value of each output.

The sum is defined to the bit: the output without a bias in fp32, plus the bias in fp32,
rounded once to the output type.  Shapes: small tiles with ragged edges (N no multiple of 4, so
elements are stored one by one), a grid of half tiles, and grids of full tiles with a last
round of half tiles, those with ragged edges too."""
import pytest
import torch

import comfy_kitchen as ck
from routes import route

pytestmark = pytest.mark.gpu

SHAPES = [(70, 37, 64, "small"), (300, 1001, 160, "small"), (4352, 4000, 64, (256, 16)), (700, 9003, 160, (0, 108)),
          (4352, 4099, 96, (256, 33))]


def _check(call, n, bias_dtype, out_dtype):
    bias = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(bias_dtype).cuda()
    plain = call(None, torch.float32)
    got = call(bias, out_dtype)
    assert torch.equal(got, (plain + bias.float()).to(out_dtype))


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bias_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,n,k,tiles", SHAPES)
def test_tile_bias(m, n, k, tiles, bias_dtype, out_dtype, hip):
    for fmt in ("mx", "nv"):
        kind, *form = route(fmt, m, n, k)
        assert kind == "small" == tiles or kind == "tiles" and tuple(form[:2]) == tiles
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x = torch.randn(m, k, generator=g, device="cuda").bfloat16()
    w = torch.randn(n, k, generator=g, device="cuda").bfloat16()
    qx, sx = ck.quantize_mxfp8(x)
    qw, sw = ck.quantize_mxfp8(w)
    _check(lambda b, o: ck.scaled_mm_mxfp8(qx, qw, sx, sw, bias=b, out_dtype=o), n, bias_dtype, out_dtype)
    one = torch.full((1,), 0.37, device="cuda")
    _check(lambda b, o: ck.scaled_mm_fp8(qx, qw, one, one, bias=b, out_dtype=o), n, bias_dtype, out_dtype)
    s = torch.full((1,), 0.01, device="cuda")
    nx, bx = ck.quantize_nvfp4(x, s)
    nw, bw = ck.quantize_nvfp4(w, s)
    _check(lambda b, o: ck.scaled_mm_nvfp4(nx, nw, s, s, bx, bw, bias=b, out_dtype=o), n, bias_dtype, out_dtype)
