"""GEMM kernels: facts that hold by construction, computed on the host from the kernels' own
headers (tests/hw/tiles.hip)."""
import pytest

from routes import library, route


@pytest.mark.parametrize("nv,tm,tn", [(0, 64, 64), (0, 128, 64), (0, 128, 96), (0, 128, 128), (0, 128, 160),
                                      (0, 128, 192), (0, 64, 128), (1, 64, 64), (1, 64, 128), (1, 128, 128),
                                      (1, 128, 192)])
def test_bias_reads_end_with_the_tile(nv, tm, tn):
    """The waves that add a tile's bias read its tn staged values, the last one included, and
    nothing past them (with four K groups, two hold no sums and must not read)."""
    assert library().ckh_tile_bias_end(nv, tm, tn) == tn


def test_every_skinny_form_is_reached():
    """No skinny kernel is compiled that no size selects."""
    for nv, fmt in enumerate(("mx", "nv")):
        seen = {route(fmt, m, n, k) for m in (1, 4, 8, 12, 16, 17, 24, 32, 33, 48, 64)
                for n in (64, 4096, 8192, 16384, 16392, 24576, 24584, 32768, 40000) for k in (512, 1024, 4096, 4128, 12288)}
        assert len({r for r in seen if r[0] == "skinny"}) == library().ckh_skinny_forms(nv)
