"""The kernels that include/hkv_device.hpp offers to callers compile as callers launch them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CALLER = r"""
#include "hkv_device.hpp"

struct Pred {
  __device__ bool operator()(uint64_t key, uint64_t score, uint64_t pattern, uint64_t threshold) const {
    return key != pattern && score >= threshold;
  }
};

void export_to(hkv_table_view v, uint64_t n, unsigned long long* count, uint64_t* keys, uint8_t* values, hipStream_t s) {
  const unsigned blocks = hkv::export_grid(n, hkv::kExportThreads);
  hipLaunchKernelGGL((hkv::export_if_kernel<Pred>), dim3(blocks), dim3(hkv::kExportThreads), 0, s, v, Pred(), 1, 2, 0, n,
                     count, keys, values, static_cast<uint64_t*>(nullptr));
}
"""


def test_callers_launch_the_export_kernel(tmp_path):
    src = tmp_path / "caller.hip"
    src.write_text(CALLER)
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-std=c++17",
                           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-fsyntax-only",
                           "-I", os.path.join(ROOT, "include"), str(src)])
