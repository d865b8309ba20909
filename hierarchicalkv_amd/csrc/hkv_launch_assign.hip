/*
 * Kernel instances of the assign family.
 */
#include "hkv_launch.hpp"

namespace hkv {
namespace {

template <bool LOCKFREE>
void launch_assign_by(int vec, const View& v, const AssignArgs& a, hipStream_t s) {
  const dim3 grid(grid_for(a.n)), block(kWave);
  if (vec == 16) {
    switch (pick_upl(v.value_bytes)) {
      case 1: hipLaunchKernelGGL((assign_kernel<16, 1, LOCKFREE>), grid, block, 0, s, v, a); break;
      case 2: hipLaunchKernelGGL((assign_kernel<16, 2, LOCKFREE>), grid, block, 0, s, v, a); break;
      case 4: hipLaunchKernelGGL((assign_kernel<16, 4, LOCKFREE>), grid, block, 0, s, v, a); break;
      default: hipLaunchKernelGGL((assign_kernel<16, 8, LOCKFREE>), grid, block, 0, s, v, a); break;
    }
  } else if (vec == 4) {
    hipLaunchKernelGGL((assign_kernel<4, 8, LOCKFREE>), grid, block, 0, s, v, a);
  } else {
    hipLaunchKernelGGL((assign_kernel<1, 8, LOCKFREE>), grid, block, 0, s, v, a);
  }
}

}  // namespace

void launch_assign(bool lockfree, int vec, const View& v, const AssignArgs& a, hipStream_t s) {
  if (lockfree)
    launch_assign_by<true>(vec, v, a, s);
  else
    launch_assign_by<false>(vec, v, a, s);
}

}  // namespace hkv
