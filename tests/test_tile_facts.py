"""Small-tile GEMMs: facts that hold by construction, computed on the host from the kernels' own
headers (tests/hw/tiles.hip)."""
import ctypes
from pathlib import Path

import pytest
import torch  # noqa: F401  (brings the HIP runtime the library links against)

LIB = Path(__file__).resolve().parent / "hw" / "libckh_hwcheck.so"


@pytest.fixture(scope="module")
def lib():
    if not LIB.exists():
        pytest.fail(f"{LIB} missing: run python comfy-kitchen_amd/build.py")
    return ctypes.CDLL(str(LIB))


@pytest.mark.parametrize("nv,tm,tn", [(0, 64, 64), (0, 128, 64), (0, 128, 96), (0, 128, 128), (0, 128, 160),
                                      (0, 128, 192), (0, 64, 128), (1, 64, 64), (1, 64, 128), (1, 128, 128),
                                      (1, 128, 192)])
def test_bias_reads_end_with_the_tile(nv, tm, tn, lib):
    """The waves that add a tile's bias read its tn staged values, the last one included, and
    nothing past them (with four K groups, two hold no sums and must not read)."""
    assert lib.ckh_tile_bias_end(nv, tm, tn) == tn
