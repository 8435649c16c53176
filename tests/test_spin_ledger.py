"""Which reductions may run together, on the CPU with made-up streams and events
(tests/cpp/spin_ledger_test.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_ledger(tmp_path):
    exe = str(tmp_path / "spin_ledger_test")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-pthread",
                    "-I", os.path.join(ROOT, "abacus-develop_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "spin_ledger_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
