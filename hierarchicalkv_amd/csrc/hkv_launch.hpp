/*
 * Choice of a kernel instance and its launch, for the kernels that come in many instances.  Each
 * family is compiled in a translation unit of its own, so that they build side by side:
 *   hkv_launch_lookup.hip   find, find*, contains, missed-keys find
 *   hkv_launch_upsert.hip   one operation of the upsert family (compiled once per operation)
 *   hkv_launch_assign.hip   assign, assign_scores, assign_values
 */
#ifndef HKV_LAUNCH_HPP_
#define HKV_LAUNCH_HPP_

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "hkv_upsert.hpp"

namespace hkv {

/* hkv_time_next_kernel: the pair of events that the calling thread's next main kernel (the one
 * kernel of a find or of an upsert-family call) is launched with.  The runtime stamps them with
 * the start and the end of that kernel's execution, so the time between them is the kernel's own,
 * without the gaps between the launches of a stream that events recorded around a call include. */
extern thread_local hipEvent_t g_time_start, g_time_stop;

template <class... KArgs, class... Args>
void launch_main(void (*kernel)(KArgs...), dim3 grid, dim3 block, hipStream_t s, Args... args) {
  if (g_time_start) {
    hipExtLaunchKernelGGL(kernel, grid, block, 0, s, g_time_start, g_time_stop, 0, args...);
    g_time_start = g_time_stop = nullptr;
  } else {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, args...);
  }
}

inline unsigned grid_for(uint64_t n) { return (unsigned)((n + kWave - 1) / kWave); }

/* 16-byte units per lane that the bulk copy keeps in registers: rows of up to 8 * UPL units (128, 256,
 * 512, 1024 bytes) go through in one pass */
inline int pick_upl(uint32_t value_bytes) {
  if (value_bytes <= 128) return 1;
  if (value_bytes <= 256) return 2;
  if (value_bytes <= 512) return 4;
  return 8;
}

/* `vec`: the unit of the row copies (lookup_unit, pick_vec, accum_unit in hkv_table.hip) */
void launch_find(int vec, const View& v, const FindArgs& a, hipStream_t s);
void launch_find_dual(int vec, const View& v, const FindArgs& a, hipStream_t s);
void launch_find_missed(int vec, const View& v, const FindArgs& a, hipStream_t s);
void launch_find_ptr(const View& v, const FindArgs& a, hipStream_t s);
void launch_contains(const View& v, const FindArgs& a, hipStream_t s);

struct UpsertForm {
  bool locked_rule; /* LOCKED slots may sit in the table: the victim scan reads key words too */
  bool bounds;      /* victims are searched through the score bounds */
  bool pair;        /* insert_and_evict: the wavefronts of a workgroup share their claims */
  bool repeats;     /* the batch may repeat keys, of which all but the first count as the EMPTY key */
};
template <int OP>
void launch_upsert(const UpsertForm& form, int vec, const View& v, const UpsertArgs& a, hipStream_t s);
extern template void launch_upsert<kOpInsertOrAssign>(const UpsertForm&, int, const View&, const UpsertArgs&, hipStream_t);
extern template void launch_upsert<kOpInsertAndEvict>(const UpsertForm&, int, const View&, const UpsertArgs&, hipStream_t);
extern template void launch_upsert<kOpFindOrInsert>(const UpsertForm&, int, const View&, const UpsertArgs&, hipStream_t);
extern template void launch_upsert<kOpAccumOrAssign>(const UpsertForm&, int, const View&, const UpsertArgs&, hipStream_t);
extern template void launch_upsert<kOpFindOrInsertPtr>(const UpsertForm&, int, const View&, const UpsertArgs&, hipStream_t);

void launch_assign(bool lockfree, int vec, const View& v, const AssignArgs& a, hipStream_t s);

}  // namespace hkv
#endif
