"""The index of repeated keys where HIP calls fail (tests/cpp/repeat_index_test.hip).  The program defines the HIP calls
itself: no GPU is used, whether there is one or not."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_index_where_calls_fail(tmp_path):
    binary = str(tmp_path / "repeat_index_test")
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-O1", "-std=c++17",
                           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                           "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "hierarchicalkv_amd", "csrc"),
                           os.path.join(HERE, "cpp", "repeat_index_test.hip"), "-o", binary])
    r = subprocess.run([binary], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout + r.stderr
