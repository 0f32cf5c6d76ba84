"""The search tile's window arithmetic on the CPU (tests/cpp/window_tests.hip, built by the package
Makefile)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BIN = os.path.join(ROOT, "simd_set_operations_amd", "cpp", "build", "window_tests")


def test_window_arithmetic():
    assert os.path.exists(BIN), "run __graft_entry__.build() (make -C simd_set_operations_amd/csrc)"
    r = subprocess.run([BIN], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0 and "0 failures" in r.stdout, r.stdout
