"""Bands per launch of the density pass by what is held and free, on the CPU
(tests/cpp/rho_bands_test.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bands(tmp_path):
    exe = str(tmp_path / "rho_bands_test")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                    "-I", os.path.join(ROOT, "abacus-develop_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "rho_bands_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
