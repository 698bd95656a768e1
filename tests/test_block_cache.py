"""The library's cache of device blocks against simulated devices (CPU only):
tests/block_cache_check.cpp over csrc/block_cache.h."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_block_cache_against_simulated_devices(tmp_path):
    exe = str(tmp_path / "block_cache_check")
    r = subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-Wextra",
                        "-I" + os.path.join(ROOT, "matrix_format_performance_amd", "csrc"),
                        os.path.join(ROOT, "tests", "block_cache_check.cpp"), "-o", exe, "-lpthread"],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
