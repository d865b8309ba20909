/*
 * Kernel instances of one operation of the upsert family: HKV_UPSERT_OP, an UpsertOp.
 */
#include "hkv_launch.hpp"

namespace hkv {
namespace {

/* BOUNDS: the victim search reads the bucket's score bounds and one or two of its score lines
 * instead of all eight (hkv_upsert.hpp).
 * R: keys per tile (hkv_lookup.hpp).
 * vec: accum_or_assign adds in units of whole elements (accum_unit); the others move rows of 16 bytes
 * and more in 16-byte units at any address, shorter ones in one or two units of the widest power of
 * two that fits (lookup_unit). */
template <int OP, int R, bool MANY, bool LOCKED_RULE, bool BOUNDS = false, int WAVES = 1, bool HOLD = false>
void launch_form(int vec, const View& v, const UpsertArgs& a, hipStream_t s) {
  constexpr uint64_t kKeys = (uint64_t)kTilesPerWave * R * WAVES;
  const dim3 grid((unsigned)((a.n + kKeys - 1) / kKeys)), block(kWave * WAVES);
  if constexpr (OP == kOpFindOrInsertPtr) { /* moves no rows */
    launch_main(upsert_kernel<OP, 16, 1, LOCKED_RULE, BOUNDS, WAVES, HOLD, R>, grid, block, s, v, a);
  } else {
    constexpr bool kAdds = OP == kOpAccumOrAssign;
    constexpr bool kFive = MANY && fits_five_waves<OP, 1, BOUNDS, HOLD, R>(); /* (rows of up to 256 bytes) */
    constexpr int kWide = kAdds ? 16 : kAny + 16;
    if (vec_bytes(vec) == 16) {
      switch (pick_upl(v.value_bytes)) {
        case 1: launch_main(upsert_kernel<OP, kWide, 1, LOCKED_RULE, BOUNDS, WAVES, HOLD, R, kFive>, grid, block, s, v, a); break;
        case 2: launch_main(upsert_kernel<OP, kWide, 2, LOCKED_RULE, BOUNDS, WAVES, HOLD, R, kFive>, grid, block, s, v, a); break;
        case 4: launch_main(upsert_kernel<OP, kWide, 4, LOCKED_RULE, BOUNDS, WAVES, HOLD, R>, grid, block, s, v, a); break;
        default: launch_main(upsert_kernel<OP, kWide, 8, LOCKED_RULE, BOUNDS, WAVES, HOLD, R>, grid, block, s, v, a); break;
      }
      return;
    }
    constexpr int kNarrow = kAdds ? 0 : kAny;
    constexpr int kUpl = kAdds ? 8 : 1; /* the others' rows have no more than two units of less than 16 bytes */
    switch (vec_bytes(vec)) {
      case 8: launch_main(upsert_kernel<OP, kNarrow + 8, kUpl, LOCKED_RULE, BOUNDS, WAVES, HOLD, R, kFive>, grid, block, s, v, a); break;
      case 4: launch_main(upsert_kernel<OP, kNarrow + 4, kUpl, LOCKED_RULE, BOUNDS, WAVES, HOLD, R, kFive>, grid, block, s, v, a); break;
      case 2: launch_main(upsert_kernel<OP, kNarrow + 2, kUpl, LOCKED_RULE, BOUNDS, WAVES, HOLD, R, kFive>, grid, block, s, v, a); break;
      default: launch_main(upsert_kernel<OP, 1, kUpl, LOCKED_RULE, BOUNDS, WAVES, HOLD, R, kFive>, grid, block, s, v, a); break;
    }
  }
}

/* insert_and_evict with `pair`: the wavefronts of a workgroup share the claims on the
 * evicted-keys output (hkv_upsert.hpp), two of 64 keys or four of 8 or 16.  Fewer keys per claim
 * queue up at the counter, more wait for each other at every trip.  2^12 keys of 64 bytes, workgroups
 * of 4 / 8 / 16 wavefronts with a key per tile: 60.5 / 63.5 / 67.4 us for the call; 2^17 of 128 bytes, two
 * keys per tile: 101.5 / 102.4 / 108.3. */
template <int OP, bool LOCKED_RULE, bool BOUNDS, int R, bool MANY = false>
void launch_upsert_for(bool pair, int vec, const View& v, const UpsertArgs& a, hipStream_t s) {
  if constexpr (OP == kOpInsertOrAssign || OP == kOpFindOrInsert) {
    /* hybrid mode: the list of slots that stay LOCKED to the end of the launch */
    if (a.held_scores) {
      launch_form<OP, R, MANY, LOCKED_RULE, BOUNDS, 1, true>(vec, v, a, s);
      return;
    }
  }
  if constexpr (OP == kOpInsertAndEvict) {
    if (pair) {
      launch_form<OP, R, MANY, LOCKED_RULE, BOUNDS, R == kTile ? 2 : 4>(vec, v, a, s);
      return;
    }
  }
  launch_form<OP, R, MANY, LOCKED_RULE, BOUNDS, 1>(vec, v, a, s);
}

/* Keys per tile.  With 8 a wavefront takes 64 keys through the victim search and the row copies one or two at
 * a time, so that a batch of a few ten thousand keys is a long chain on part of the chip; with fewer
 * keys per tile the chain is shorter, and every step is issued for fewer keys at once, which is what
 * costs once the chip is full anyway.  (Registers hardly come into it: insert_or_assign with bounds is
 * compiled to 124 with eight, 97 or 96 with two, 95 with one, i.e. 4, 4 or 5, and 5 wavefronts per SIMD; the table was
 * measured while two always had 97 and four.)  us per call,
 * eight / two / one, LRU, rows of 64 bytes; the order is the same for 256:
 *            capacity 2^24, full, half of the keys found          ... 95 % found           a third full, all found
 *            insert_or_assign    insert_and_evict      insert_or_assign   insert_and_evict   insert_or_assign
 *   2^12     29 / 15 / 13        38 / 23 / 20          29 / 15 / 13       37 / 23 / 20       14 /  9 /  8
 *   2^14     30 / 18 / 16        42 / 25 / 24          33 / 20 / 17       42 / 26 / 25       14 / 11 / 10
 *   2^15     38 / 25 / 22        48 / 31 / 33          40 / 25 / 23       49 / 34 / 33       16 / 12 / 12
 *   2^16     43 / 29 / 31        63 / 45 / 53          43 / 30 / 31       65 / 45 / 53       19 / 15 / 18
 *   2^17     71 / 55 / 54        92 / 76 / 88          59 / 49 / 51       89 / 73 / 86       25 / 25 / 31
 *   2^18    104 / 93 / 96       120 / 117 / 144        74 / 76 / 82       74 / 92 / 130      36 / 44 / 55
 *   2^20    345 / 333 / 348     431 / 437 / 531       173 / 211 / 238    205 / 267 / 364    142 / 160 / 217
 * The line at 2^18: with many new keys per bucket two per tile are far ahead there (capacity 2^21, all keys new,
 * 216 / 145; accum_or_assign, half of them, 153 / 117); what they lose where nearly all keys are found, on a
 * table that only has been offered nine tenths of its slots for instance, is less (accum_or_assign of keys
 * that are all there or change nothing: 35 / 41).  A batch that came with repeated ids (`repeats`) has many of
 * its keys crossed off and takes eight above 2^17: 2^18 keys 133 / 147 / 156 with the passes over the ids (three launches
 * per call then, one now: 116 with eight).  Not so the pointer overload, which moves no rows: eight are better for it where
 * most ids repeat or are found (200 000 Zipf ids 36 / 43), and far worse where few do (140 000 uniform ones, most of
 * them new to a full table, 150 / 107).
 * Two keys per tile in more wavefronts than four per SIMD (256 CUs, 1024 SIMDs: 2^16 keys) take the instance that leaves room
 * for a fifth, others the one that does not have to.  insert_or_assign, half of the keys new, us with four / five:
 *                        34 000         60 000         2^16           68 000         80 000         100 000
 *   rows of  40 bytes    22.9 / 23.1    29.7 / 29.9    31.1 / 31.3    32.6 / 31.9    36.7 / 35.1    42.1 / 41.7
 *   rows of 256 bytes    23.7 / 24.0    30.3 / 30.4    31.6 / 31.7    33.2 / 32.3    37.7 / 35.4    43.4 / 42.9 */
constexpr uint64_t kFourWaves = (uint64_t)1024 * 4 * kTilesPerWave * 2;
template <int OP, bool BOUNDS>
void launch_by_size(bool pair, bool repeats, int vec, const View& v, const UpsertArgs& a, hipStream_t s) {
  if (a.n <= (UINT64_C(1) << (BOUNDS ? 15 : 14)))
    launch_upsert_for<OP, false, BOUNDS, 1>(pair, vec, v, a, s);
  else if (a.n <= kFourWaves)
    launch_upsert_for<OP, false, BOUNDS, 2>(pair, vec, v, a, s);
  else if (a.n <= (UINT64_C(1) << (BOUNDS && !(repeats && OP != kOpFindOrInsertPtr) ? 18 : 17)))
    launch_upsert_for<OP, false, BOUNDS, 2, true>(pair, vec, v, a, s);
  else
    launch_upsert_for<OP, false, BOUNDS, kTile>(pair, vec, v, a, s);
}

}  // namespace

template <int OP>
void launch_upsert(const UpsertForm& form, int vec, const View& v, const UpsertArgs& a, hipStream_t s) {
  if (form.locked_rule)
    launch_upsert_for<OP, true, false, kTile>(form.pair, vec, v, a, s);
  else if (form.bounds)
    launch_by_size<OP, true>(form.pair, form.repeats, vec, v, a, s);
  else
    launch_by_size<OP, false>(form.pair, form.repeats, vec, v, a, s);
}
template void launch_upsert<HKV_UPSERT_OP>(const UpsertForm&, int, const View&, const UpsertArgs&, hipStream_t);

}  // namespace hkv
