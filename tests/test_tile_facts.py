"""GEMM kernels: facts that hold by construction, computed on the host from the kernels' own
headers (tests/hw/tiles.hip)."""
import ctypes

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


@pytest.mark.parametrize("m,n,k,want", [
    (25, 8688, 1024, (4, 2, 1, 32)), (32, 9688, 2624, (4, 2, 1, 32)), (24, 10240, 5120, (4, 2, 1, 32)),
    (32, 16384, 2048, (4, 2, 1, 32)), (18, 16392, 4096, (2, 1, 1, 32)), (29, 20408, 6880, (4, 1, 1, 32)),
    (17, 24576, 4128, (4, 1, 1, 32)), (32, 30000, 4096, (2, 2, 1, 32)), (52, 19808, 512, (2, 1, 2, 64)),
    (33, 16392, 1248, (2, 1, 2, 64)), (64, 24576, 1024, (2, 1, 2, 64)), (64, 32768, 512, (2, 2, 2, 64)),
    (40, 40000, 3072, (2, 2, 2, 64))])
def test_few_rows_short_k_or_narrow_take_the_skinny_kernel(m, n, k, want):
    """Where the small tiles measured slower than the skinny kernel, in the form that measured best."""
    assert route("mx", m, n, k)[:5] == ("skinny", *want)


@pytest.mark.parametrize("m,n,k,want", [
    (32, 16384, 3072, (64, 64)), (17, 10248, 5120, (64, 64)), (17, 24576, 4224, (64, 128)),
    (20, 32768, 4128, (64, 128)), (64, 8192, 512, (64, 64)), (33, 16384, 32, (64, 64)),
    (48, 18432, 1280, (64, 128)), (64, 32768, 640, (64, 128))])
def test_few_rows_small_tiles(m, n, k, want):
    assert route("mx", m, n, k) == ("small", *want)


@pytest.mark.parametrize("m,n,k,want", [
    (50, 9232, 928, ("skinny", 4, 2, 2, 0, 0)), (64, 30000, 992, ("skinny", 4, 2, 2, 0, 0)),
    (33, 8192, 32, ("skinny", 4, 2, 2, 0, 0)), (33, 8192, 768, ("small", 64, 64)), (40, 8200, 1056, ("small", 64, 64)),
    (64, 17001, 1024, ("small", 64, 128)), (32, 9000, 1024, ("skinny", 4, 2, 1, 0, 0))])
def test_nvfp4_few_rows(m, n, k, want):
    """Short rows that do not start on a cache line measured slower in small tiles."""
    assert route("nv", m, n, k) == want


@pytest.mark.parametrize("m,n,k,want", [
    (1024, 4368, 13728, ("split", 3, 72, 4)), (848, 560, 7072, ("split", 7, 16, 2)),
    (691, 1312, 5824, ("small", 64, 64)), (1024, 4336, 4096, ("small", 128, 160))])
def test_ragged_rows_shared_by_many_tiles(m, n, k, want):
    """Rows that do not start on a cache line cost small tiles more, also with over six of them
    along m: long K splits there, as it measured faster."""
    assert route("mx", m, n, k) == want


@pytest.mark.parametrize("m,n,k,want", [
    (200, 792, 8704, ("split", 7, 5, 2)), (146, 576, 7040, ("split", 7, 4, 2)), (200, 792, 4096, ("small", 64, 64))])
def test_nvfp4_narrow_layers_with_long_k_split(m, n, k, want):
    assert route("nv", m, n, k) == want


@pytest.mark.parametrize("rows,cols,fast", [(230, 1856, False), (1, 3072, False), (1023, 3072, False), (1025, 3072, True),
                                            (16, 64, True), (240, 1856, True)])
def test_nvfp4_quantize_of_padded_rows(rows, cols, fast):
    """Small inputs padded in rows take the general kernel, which measured faster there."""
    f = library().ckh_nv_quantize_fast_rows
    f.argtypes = [ctypes.c_int64] * 3
    assert f(-(-rows // 16) * 16, rows, cols) == fast
