/*
 * Kernel instances of the lookups.
 */
#include "hkv_launch.hpp"

namespace hkv {
namespace {

/* the part of a call from key `first` on, at most `most` keys of it */
FindArgs part_of(const View& v, const FindArgs& a, uint64_t first, uint64_t most) {
  FindArgs p = a;
  p.keys += first;
  if (p.out_values) p.out_values += first * v.value_bytes;
  if (p.out_ptrs) p.out_ptrs += first;
  if (p.founds) p.founds += first;
  if (p.out_scores) p.out_scores += first;
  p.n = a.n - first < most ? a.n - first : most;
  return p;
}

template <int MODE, int R, bool DUAL, int WAVES, bool MISSED>
void launch_one(int vec, const View& v, const FindArgs& a, hipStream_t s) {
  constexpr uint64_t kKeys = (uint64_t)kTilesPerWave * R * WAVES;
  const dim3 grid((unsigned)((a.n + kKeys - 1) / kKeys)), block(kWave * WAVES);
  if constexpr (MODE == kLookupValues) {
    switch (vec) {
      case kAny + 16: launch_main(lookup_kernel<MODE, kAny + 16, DUAL, WAVES, R, MISSED>, grid, block, s, v, a); return;
      case kAny + 8: launch_main(lookup_kernel<MODE, kAny + 8, DUAL, WAVES, R, MISSED>, grid, block, s, v, a); return;
      case kAny + 4: launch_main(lookup_kernel<MODE, kAny + 4, DUAL, WAVES, R, MISSED>, grid, block, s, v, a); return;
      case kAny + 2: launch_main(lookup_kernel<MODE, kAny + 2, DUAL, WAVES, R, MISSED>, grid, block, s, v, a); return;
      case 1: launch_main(lookup_kernel<MODE, 1, DUAL, WAVES, R, MISSED>, grid, block, s, v, a); return;
    }
  }
  launch_main(lookup_kernel<MODE, 16, DUAL, WAVES, R, MISSED>, grid, block, s, v, a);
}

/* One launch for all but the longest batches: two keys per tile are four threads per key, 2^31 of them at
 * 2^29 keys.  (The missed-keys form has one thread per key, and its 32-bit indices end before that matters.) */
template <int MODE, int R, bool DUAL = false, int WAVES = 1, bool MISSED = false>
void launch_lookup_by(int vec, const View& v, const FindArgs& a, hipStream_t s) {
  if constexpr (MISSED) {
    launch_one<MODE, R, DUAL, WAVES, MISSED>(vec, v, a, s);
  } else {
    constexpr uint64_t kMost = kLaunchThreads / (kTile / R);
    for (uint64_t first = 0; first < a.n; first += kMost)
      launch_one<MODE, R, DUAL, WAVES, MISSED>(vec, v, part_of(v, a, first, kMost), s);
  }
}

/* Keys per tile.  A wavefront of 64 keys (R = 8) was compiled to 114 registers, four of them fit on a SIMD,
 * and a tile does much of its work on its 8 keys one after the other; with 2 keys per tile it is 48
 * registers, eight wavefronts, and a quarter of the chain (with 1, 33).  us per call (hits 7/8, cold):
 *   keys     row        R = 8    2      1
 *   2^20    256 bytes    119    112    115
 *   2^20     32           73     68     84
 *   2^18    512           55     51     49.5
 *   2^15    256           12.2    7.8    7.8
 *   3001     64           10.1    5.3    4.6
 *   500     256            9.6    4.6    3.8
 *   2^20   no rows (contains)  51  46.5  58
 * One key per tile where that leaves the chip room (a quarter of its 8192 wave slots at 2^14 keys)
 * or where the rows outweigh the probes.  us per call with two / one (7/8 found):
 *   row         171 667 keys     500 000 keys
 *   256 bytes   20.6 / 21.8      52.4 / 54.3
 *   320         27.1 / 27.3      68.9 / 68.9
 *   400         33.5 / 33.0      86.3 / 84.9
 *   480         37.2 / 36.0      97.0 / 93.6 */
template <int MODE>
void launch_lookup(int vec, const View& v, const FindArgs& a, hipStream_t s) {
  if (a.n <= (UINT64_C(1) << 14) || (MODE == kLookupValues && v.value_bytes >= 384))
    launch_lookup_by<MODE, 1>(vec, v, a, s);
  else
    launch_lookup_by<MODE, 2>(vec, v, a, s);
}

}  // namespace

void launch_find(int vec, const View& v, const FindArgs& a, hipStream_t s) { launch_lookup<kLookupValues>(vec, v, a, s); }
void launch_find_ptr(const View& v, const FindArgs& a, hipStream_t s) { launch_lookup<kLookupPtr>(16, v, a, s); }
void launch_contains(const View& v, const FindArgs& a, hipStream_t s) { launch_lookup<kLookupContains>(16, v, a, s); }
void launch_find_dual(int vec, const View& v, const FindArgs& a, hipStream_t s) {
  launch_lookup_by<kLookupValues, 2, true>(vec, v, a, s);
}
/* 16 wavefronts per workgroup (see lookup_kernel) */
void launch_find_missed(int vec, const View& v, const FindArgs& a, hipStream_t s) {
  launch_lookup_by<kLookupValues, kTile, false, 16, true>(vec, v, a, s);
}

}  // namespace hkv
