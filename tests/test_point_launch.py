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
    L.point_total.argtypes = [C.c_int, C.c_int, C.c_int, C.c_int, C.c_void_p]
    return L


@pytest.mark.parametrize("per", [1, 4, 16, 64])
@pytest.mark.parametrize("count", [1, 7, 8, 9, 6143, 6144, 6145, 1 << 20, (1 << 31) - 6145, (1 << 31) - 6144,
                                   (1 << 31) - 255, (1 << 31) - 1])
def test_every_query_is_walked_once(lib, count, per):
    """768 blocks of eight waves take each query once, up to the largest count
    (an int that walks by 6 144 passes 2^31 within the last 6 144 queries)."""
    last = C.c_longlong()
    assert lib.point_total(count, 8, per, 768, C.byref(last)) == count
    assert last.value == count - 1


def test_lanes_of_a_query(lib):
    """Few queries keep the whole wave; many samples do; fewer lanes come with
    more queries and fewer samples."""
    assert all(lib.lanes_of(s, 1) == 64 for s in (1, 8, 64, 1024))
    assert all(lib.lanes_of(s, (1 << 31) - 1) == 64 for s in (257, 1024, 2049, 1 << 20))
    for samples in (1, 2, 5, 16, 17, 63, 64, 65, 200, 256):
        lanes = [lib.lanes_of(samples, c) for c in (1, 2047, 2048, 8192, 32768, 163840, 1 << 20, (1 << 31) - 1)]
        assert set(lanes) <= {64, 16, 4, 1} and lanes == sorted(lanes, reverse=True)
        assert lanes[-1] * 16 >= samples
    assert [lib.lanes_of(s, 1 << 20) for s in (1, 16, 17, 64, 65, 256, 257)] == [1, 1, 4, 4, 16, 16, 64]
