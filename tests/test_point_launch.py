"""Launch arithmetic of the point prefilter (CPU, no GPU): the header that the
kernel runs, built for the host."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("pt") / "libpoint_launch.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Werror", "-fsanitize=undefined",
                    "-fsanitize-undefined-trap-on-error",
                    str(ROOT / "tests" / "cpp" / "point_launch_host.cpp"), "-o", str(so)],
                   check=True, capture_output=True)
    L = C.CDLL(str(so))
    L.point_total.restype = C.c_longlong
    L.point_total.argtypes = [C.c_int, C.c_int, C.c_int, C.c_void_p]
    return L


@pytest.mark.parametrize("count", [1, 7, 8, 9, 6143, 6144, 6145, 1 << 20, (1 << 31) - 6145, (1 << 31) - 6144,
                                   (1 << 31) - 255, (1 << 31) - 1])
def test_every_query_is_walked_once(lib, count):
    """768 blocks of eight waves take each query once, up to the largest count
    (an int that walks by 6 144 passes 2^31 within the last 6 144 queries)."""
    last = C.c_longlong()
    assert lib.point_total(count, 8, 768, C.byref(last)) == count
    assert last.value == count - 1
