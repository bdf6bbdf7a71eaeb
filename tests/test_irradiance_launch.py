"""Launch arithmetic of the irradiance (CPU, no GPU): the header that the kernel
runs, built for the host, against exact integers at the limits that the entry
points accept."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("irr") / "libirradiance_launch.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Werror", "-fsanitize=undefined",
                    "-fsanitize-undefined-trap-on-error",
                    str(ROOT / "tests" / "cpp" / "irradiance_launch_host.cpp"), "-o", str(so)],
                   check=True, capture_output=True)
    L = C.CDLL(str(so))
    L.fold_walk.restype = C.c_longlong
    L.fold_walk.argtypes = [C.c_int, C.c_int, C.c_int, C.c_int, C.c_void_p]
    L.grids.argtypes = [C.c_int, C.c_int, C.c_void_p]
    return L


@pytest.mark.parametrize("size", [1, 2, 3, 2364, 2365, 3344, 3345, 4095, 4096])
def test_grids_stay_within_the_launch_limits(lib, size):
    """Every size the entry points accept: less than 2^32 threads along x and
    2^16 blocks along y, a block of 1 024 threads for each orbit of three axes,
    a wave of 64 (four a block) for each texel of six faces."""
    g = (C.c_uint * 4)()
    lib.grids(size, 4, g)
    half = (size + 1) // 2
    assert (g[0], g[1]) == (half, 3 * half) and g[0] * 1024 < 1 << 32 and g[1] < 1 << 16
    assert g[3] == 6 and 4 * g[2] >= size * size > 4 * (g[2] - 1) and g[2] * 256 < 1 << 32


# (azimuths, polar samples): the smallest, ragged ones, the reference's 300 x
# 150, an 8 x 128 and a 64 x 1024 source at 100 000 azimuths (2.5e9 steps, past
# 2^31), and a handle of 512 x 256 at 600 000 and 2 000 000.
@pytest.mark.parametrize("theta,phi,stride", [(2, 1, 16), (8, 4, 16), (136, 7, 16), (300, 150, 16), (2050, 1025, 16),
                                              (100000, 1600000, 16 * 9973), (600000, 300000, 16 * 9973),
                                              (2000000, 1000000, 16 * 99991)])
def test_every_step_of_an_orbit_is_walked(lib, theta, phi, stride):
    """Waves 0..15 take each step of an orbit once (in strides of 16; the largest
    counts are walked in longer strides): the number of steps and the last one."""
    ts, ps = (theta + 7) // 8, (phi + 7) // 8
    total = ts * ps
    last = (C.c_int * 2)()
    for wave in (0, 1, 7, 15):
        n = lib.fold_walk(wave, stride, ts, ps, last)
        want = 0 if wave >= total else (total - 1 - wave) // stride + 1
        assert n == want, (wave, n, want)
        if n:
            step = wave + (want - 1) * stride
            assert (last[0], last[1]) == (step // ts, step % ts)
