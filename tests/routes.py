"""Which kernel a GEMM call runs, asked of the dispatch rules themselves (csrc/dispatch.h through
tests/hw/tiles.hip, on the host).  A test that is about one kernel asserts it here."""
import ctypes
import functools
from pathlib import Path

import pytest
import torch  # noqa: F401  (brings the HIP runtime the library links against)

LIB = Path(__file__).resolve().parent / "hw" / "libckh_hwcheck.so"
KINDS = {0: ("skinny", 5), 1: ("small", 2), 2: ("split", 3), 3: ("tiles", 3)}
CUS = 256  # an MI355X's


@functools.lru_cache(1)
def library() -> ctypes.CDLL:
    if not LIB.exists():
        pytest.fail(f"{LIB} missing: run python comfy-kitchen_amd/build.py")
    lib = ctypes.CDLL(str(LIB))
    lib.ckh_route.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_int] * 2 + [ctypes.c_void_p]
    return lib


def route(fmt: str, m: int, n: int, k: int, workspace: bool = True, cus: int = CUS) -> tuple:
    """("skinny", waves, weight tiles, activation tiles, activation rows, code rows),
    ("small", rows, columns), ("split", ranges, stages or groups per range, 4 whole or 2 half tiles)
    or ("tiles", whole tiles, tiles run as halves, prefetch workgroups).  fmt: "mx" (MXFP8 and
    per-tensor FP8) or "nv".  workspace: the wrappers bring one wherever K can split."""
    out = (ctypes.c_int * 6)()
    name, count = KINDS[library().ckh_route(int(fmt == "nv"), m, n, k, int(workspace), cus, out)]
    return (name, *out[:count])
