"""The batched prefilter's grid (CPU, no GPU): every setting the tuning accepts
gives each CU a block."""
import ctypes as C
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_every_cu_has_a_block(tmp_path):
    so = tmp_path / "libbatch_launch.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Werror",
                    str(ROOT / "tests" / "cpp" / "batch_launch_host.cpp"), "-o", str(so)], check=True,
                   capture_output=True)
    f = C.CDLL(str(so)).blocks_of
    for cus in (1, 32, 256):
        got = [f(cus, w, 8) for w in range(4, 33)]
        assert got == sorted(got) and got[0] == cus and all(b >= cus for b in got)
        assert all(f(cus, w, 8) == cus * w // 8 for w in range(8, 33))
