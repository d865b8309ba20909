"""The host's bookkeeping of what a load sample would read (tests/cpp/growth_test.cpp), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hierarchicalkv_amd", "csrc")


def test_bookkeeping_of_the_load(tmp_path):
    binary = str(tmp_path / "growth_test")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-I", CSRC, os.path.join(HERE, "cpp", "growth_test.cpp"),
                           "-o", binary])
    r = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout
