/*
 * Read-only lookups: find (value copy), find* (row pointer), contains, and
 * the missed-keys variant of find.  One 64-lane wavefront per workgroup, R keys
 * per 8-lane tile (8R per wavefront).
 *
 * Replaces lookup_kernel_with_io_pipeline_v1 (lookup.cuh:119-378),
 * lookup_ptr_kernel_with_pipeline / tlp_lookup_ptr_kernel_with_filter
 * (lookup_ptr.cuh:25-374) and the contains kernels (contains.cuh:46-216).
 * No slot locks are taken: the API-level group lock keeps writers out, as in
 * the reference (group_lock.cuh:43-56).
 *
 * Phases of a wavefront
 *   own    lane 8t + r (r < R) loads its key, hashes it and stages (key, bucket, digest) in LDS;
 *   probe  tile t (8 lanes) probes the key of lane 8t + r in round r < R: lane j loads
 *          16 of the 128 digest bytes, so a tile reads one whole 128-byte line
 *          per round; the rounds are issued back to back, R KB of digests in flight per wavefront;
 *   verify every digest match is checked against the 8-byte key, the first
 *          lane's candidates first and the others only if those were not it;
 *          the hit slot goes to LDS;
 *   copy   the found keys are listed in LDS, and the whole wavefront copies their rows, one unit per
 *          lane and step, so the output side is written in coalesced pieces of up to 1 KB.
 * Bound by random 128-byte lines (a digest line, about 1.2 key lines and the row per key): 528 MB in and
 * 237 MB out of the L2s in 113.5 us for 2^20 keys, 7/8 found, rows of 256 bytes, capacity 2^26 (6.7 TB/s; the
 * 64 MB of digests stay in the Infinity Cache).  How many keys a tile takes is
 * what matters most beside that (launch_lookup in hkv_launch_lookup.hip).
 */
#ifndef HKV_LOOKUP_HPP_
#define HKV_LOOKUP_HPP_

#include "hkv_common.hpp"

namespace hkv {

struct FindArgs {
  const uint64_t* keys;
  uint8_t* out_values;     /* find */
  void** out_ptrs;         /* find* */
  uint8_t* founds;         /* may be null for the missed-keys variant */
  uint64_t* out_scores;    /* optional */
  uint64_t* missed_keys;   /* missed-keys variant */
  int32_t* missed_indices;
  int32_t* missed_size;
  uint64_t n;
};

/*
 * Keys per wavefront.  Tile t owns the keys of its lanes 0 .. R-1, R = 8 being the full 64 keys of
 * a wavefront: the key of lane 8t + r is number t * R + r of the wavefront, and lanes 8t + R and
 * above own none.  What is staged in LDS is indexed by lane.  A smaller R spreads a batch over
 * more wavefronts: a tile handles its R keys one after the other where it cannot overlap them.
 */
template <int R>
__device__ __forceinline__ uint64_t key_of_lane(uint64_t wave, int lane) {
  if constexpr (R == kTile) return wave * kWave + lane;
  return wave * (kTilesPerWave * R) + (uint32_t)(lane >> 3) * R + (lane & (kTile - 1));
}
template <int R>
__device__ __forceinline__ bool lane_owns_key(int lane) {
  return R == kTile || (lane & (kTile - 1)) < R;
}
/*
 * Probe the keys staged in s_meta.  On return (after the caller's barrier)
 * s_slot[k] is the table slot of key k or -1.  WRITER selects the writers'
 * probe, which runs while other wavefronts change the table:
 *   - s_em[k][j] (when given) receives lane j's 16-bit mask of EMPTY digests of
 *     key k's bucket, bit p for byte 16j+p, so the 8 masks of a key read back
 *     as one 128-bit mask in slot order;
 *   - a candidate slot whose key word reads LOCKED may be this very key under
 *     another tile's lock, so s_unsure[k] is raised and the writer settles the
 *     question with a second, coherent probe of its own (tile_reprobe).
 */
template <bool WRITER, bool TWO_STEP, int R = kTile>
__device__ __forceinline__ void probe_wave(const View& v, const KeyMeta* s_meta,
                                           int64_t* s_slot,
                                           uint16_t (*s_em)[kTile],
                                           uint8_t* s_unsure, int lane) {
  const int tile = lane >> 3, j = lane & 7;
  uint4 dg[R];
  uint32_t bkt[R];
  uint32_t inf[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const KeyMeta m = s_meta[tile * kTile + r];
    bkt[r] = m.bkt;
    inf[r] = m.info;
    dg[r] = make_uint4(0, 0, 0, 0);
    if (m.info & 0x100u)
      dg[r] = *reinterpret_cast<const uint4*>(v.digests + (uint64_t)m.bkt * kBucketSize + j * 16);
  }
  /* TWO_STEP: candidates are verified in two steps.  An 8-byte key load costs a whole
   * 128-byte line of memory traffic, a key that is present has one true candidate, and a
   * false 8-bit match turns up in every second bucket: so step 1 fetches only the
   * candidates of one lane of the tile (a lane's 16 slots share one key line), the one
   * where the key most likely is, and the other lanes' candidates are fetched in step 2
   * only for the keys step 1 did not find: 1.03 to 1.27 key lines per key that is present
   * (keys that went into a free slot / into a victim's slot) instead of 1.44.  The lookups
   * and the kernels that move rows use it; erase and lock_keys, which move little besides
   * the probe and are bound by their dependent round trips, take all candidates at once. */
  uint32_t cm[R];       /* this lane's digest matches, bw order */
  uint32_t later[R];     /* lanes of the tile whose candidates wait for step 2 */
  uint64_t k0[R], k1[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const bool valid = inf[r] & 0x100u;
    const uint32_t d = inf[r] & 0xFFu;
    cm[r] = valid ? match16(dg[r], d * 0x01010101u) : 0u;
    if (WRITER && s_em != nullptr)
      s_em[tile * kTile + r][j] =
          (uint16_t)(valid ? match16_natural(dg[r], v.empty_digest * 0x01010101u) : 0u);
    const uint32_t lanes = TWO_STEP ? tile_ballot(cm[r] != 0, tile) : 0u;
    /* step 1 takes the first lane with a candidate at or after the lane of the key's start
     * slot, going round: an insert takes the first free slot from there (the reference's
     * probe order, kernel_utils.cuh:636-643), so that is where the key most likely is */
    const uint32_t sl = inf[r] >> 20; /* start slot / 16 */
    const uint32_t turned = ((lanes >> sl) | (lanes << (kTile - sl))) & 0xFFu;
    const uint32_t first = (uint32_t)(__ffs(turned) - 1 + sl) & (kTile - 1);
    later[r] = lanes & ~(1u << first);
    const uint64_t* kb = v.keys + (uint64_t)bkt[r] * kBucketSize + j * 16;
    k0[r] = v.empty_key;
    k1[r] = v.empty_key;
    if (cm[r] && !((later[r] >> j) & 1u)) {
      k0[r] = kb[bw_to_pos(__ffs(cm[r]) - 1)];
      const uint32_t rest = cm[r] & (cm[r] - 1);
      if (rest) k1[r] = kb[bw_to_pos(__ffs(rest) - 1)];
    }
  }
  /* checks the candidates of this lane for key r against the fetched words (the third and
   * later candidates of a lane, rare, are loaded here) */
  auto check = [&](int r) {
    const int kk = tile * kTile + r;
    const uint64_t key = s_meta[kk].key;
    const uint64_t slot0 = (uint64_t)bkt[r] * kBucketSize + j * 16;
    uint32_t m = cm[r];
    int hit = -1;
    bool unsure = false;
    int c = 0;
    while (m) {
      const uint32_t p = bw_to_pos(__ffs(m) - 1);
      m &= m - 1;
      const uint64_t kx = c == 0 ? k0[r] : (c == 1 ? k1[r] : v.keys[slot0 + p]);
      c++;
      if (kx == key) {
        hit = (int)p;
        break;
      }
      if (WRITER && kx == v.locked_key) unsure = true;
    }
    if (hit >= 0)
      s_slot[kk] = (int64_t)(slot0 + hit);
    else if (WRITER && unsure)
      s_unsure[kk] = 1;
    return hit >= 0;
  };
  bool more = false;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const bool mine = cm[r] && !((later[r] >> j) & 1u);
    const bool hit = mine && check(r);
    if (TWO_STEP) {
      if (tile_ballot(hit, tile)) later[r] = 0;
      more |= later[r] != 0;
    }
  }
  if (TWO_STEP && __ballot(more)) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      if ((later[r] >> j) & 1u) {
        const uint64_t* kb = v.keys + (uint64_t)bkt[r] * kBucketSize + j * 16;
        k0[r] = kb[bw_to_pos(__ffs(cm[r]) - 1)];
        const uint32_t rest = cm[r] & (cm[r] - 1);
        if (rest) k1[r] = kb[bw_to_pos(__ffs(rest) - 1)];
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
      if ((later[r] >> j) & 1u) check(r);
  }
}

/* the writers' probes (upsert and assign families): they move rows, like find */
constexpr bool kTwoStepWriters = true;

/* the 16 digest bytes of lane j of a tile, read past the caches */
__device__ __forceinline__ uint4 ld_digests16(const View& v, uint32_t bkt, int j) {
  const uint64_t off = (uint64_t)bkt * kBucketSize + j * 16;
  if (v.capacity < (UINT64_C(1) << 32)) return ld_u128_at(v.digests, v.capacity, off);
  const uint32_t* dp = reinterpret_cast<const uint32_t*>(v.digests + off);
  uint4 d;
  d.x = ld_u32(dp + 0);
  d.y = ld_u32(dp + 1);
  d.z = ld_u32(dp + 2);
  d.w = ld_u32(dp + 3);
  return d;
}

/*
 * Second opinion for a writer, by the 8-lane tile that owns the key, with
 * coherent loads: returns the slot of the key, -1 when the key is not in the
 * bucket, or -2 when a digest-matching slot is LOCKED right now (ask again).
 * `em` receives the lane's fresh mask of EMPTY digests (bit p for byte 16j+p).
 */
__device__ __forceinline__ int64_t tile_reprobe(const View& v, uint64_t key,
                                                uint32_t bkt, uint32_t digest,
                                                int tile, int j, uint32_t& em) {
  const uint4 d = ld_digests16(v, bkt, j);
  em = match16_natural(d, v.empty_digest * 0x01010101u);
  uint32_t m = match16(d, digest * 0x01010101u);
  const uint64_t slot0 = (uint64_t)bkt * kBucketSize + j * 16;
  int hit = -1;
  bool locked = false;
  while (m) {
    const uint32_t p = bw_to_pos(__ffs(m) - 1);
    m &= m - 1;
    const uint64_t kx = ld_u64(v.keys + slot0 + p);
    if (kx == key) {
      hit = (int)p;
      break;
    }
    if (kx == v.locked_key) locked = true;
  }
  const uint32_t hits = tile_ballot(hit >= 0, tile);
  const uint32_t locks = tile_ballot(locked, tile);
  if (hits) {
    const int jl = __ffs(hits) - 1;
    return (int64_t)tile_bcast((uint32_t)hit, tile, jl) + (int64_t)bkt * kBucketSize + jl * 16;
  }
  return locks ? -2 : -1;
}

/* Lane-owned part shared by all probing kernels: load, hash, stage.  Lanes without a key pass i >= n. */
__device__ __forceinline__ uint64_t stage_keys(const View& v,
                                               const uint64_t* keys, uint64_t n,
                                               uint64_t i, KeyMeta* s_meta,
                                               int64_t* s_slot, int lane) {
  uint64_t key = v.empty_key;
  if (i < n) key = keys[i];
  const bool valid = (i < n) && !is_reserved_key(v, key);
  uint32_t bkt = 0, start = 0, digest = 0;
  locate(v, key, bkt, start, digest);
  KeyMeta m;
  m.key = key;
  m.bkt = bkt;
  m.info = digest | (valid ? 0x100u : 0u) | (start << 16);
  s_meta[lane] = m;
  s_slot[lane] = -1;
  return key;
}

/* First pass of a dual-bucket find (dual_bucket_lookup.cuh:25-140): the keys
 * staged by stage_keys get their first bucket and the dual-mode digest. */
__device__ __forceinline__ void restage_first_bucket(const View& v, KeyMeta* s_meta, int lane) {
  KeyMeta m = s_meta[lane];
  if (m.info & 0x100u) {
    const DualLoc L = locate_dual(v, m.key);
    m.bkt = L.bkt[0];
    m.info = L.digest | 0x100u | (L.start[0] << 16);
    s_meta[lane] = m;
  }
}
/* Second pass of a dual-bucket find: the keys of the wavefront that b1 did not
 * hold are staged again with their second bucket; the others are switched off. */
__device__ __forceinline__ void restage_second_bucket(const View& v, KeyMeta* s_meta,
                                                      const int64_t* s_slot, int lane) {
  KeyMeta m = s_meta[lane];
  const bool again = (m.info & 0x100u) && s_slot[lane] < 0;
  if (again) {
    const DualLoc L = locate_dual(v, m.key);
    m.bkt = L.bkt[1];
    m.info = L.digest | 0x100u | (L.start[1] << 16);
  } else {
    m.info &= ~0x100u;
  }
  s_meta[lane] = m;
}


enum LookupMode { kLookupValues = 0, kLookupPtr = 1, kLookupContains = 2 };

/* Where a found key's row is and where it goes, in one word: the slot (buckets_num < 2^31, so below
 * 2^38) and the key's number in its wavefront. */
constexpr int kFoundShift = 56;
constexpr uint64_t kFoundSlot = (UINT64_C(1) << kFoundShift) - 1;
/* a key that was not found: reads slot 0's row, and its place is past the end of any wavefront's rows (a row is at
 * most 2^20 bytes) */
constexpr uint64_t kListedMiss = UINT64_C(0xFF) << kFoundShift;

/* Where the rows of the table are; an address is one multiply-add in the first case (slot numbers fit 32 bits
 * there).  A lane past the end of the list reads a row that the caches have: the first key's; slot 0's, in
 * HBM; or, so that it does not go over the host link, the first digests (as an address beside the two others
 * these cost 3 of 84 us on a table with rows in both places). */
enum RowsIn { kRowsHbm, kRowsBoth, kRowsHost };

/* The rows of the `count` found keys listed in `found` -> their places in `out`, where key `base` is the first of
 * the wavefront. */
template <int VEC, int R, int WHERE, int kB>
__device__ __forceinline__ void copy_units(const View& v, const uint64_t* found, uint32_t count, uint32_t units,
                                           uint8_t* out, uint64_t base, uint64_t n, int lane) {
  using T = typename VecType<VEC>::type;
  constexpr uint32_t kKeys = kTilesPerWave * R;
  constexpr uint32_t kPast = 0x80000000u; /* an offset that is past the end of any wavefront's rows */
  const uint32_t total = units * count;
  const uint64_t rows_here = n - base < kKeys ? n - base : kKeys;
  const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc(
      out + base * v.value_bytes, 0, (uint32_t)(rows_here * v.value_bytes), 0x00020000);
  /* (found key, unit) of this lane's next step; a step moves 64 units on */
  uint32_t kk = (uint32_t)lane / units, c = (uint32_t)lane % units;
  const uint32_t kk_step = kWave / units, c_step = kWave % units;
  for (uint32_t idx0 = lane; idx0 < total; idx0 += kWave * kB) {
    T buf[kB];
    uint32_t at[kB];
#pragma unroll
    for (int b = 0; b < kB; b++) {
      const bool inside = kk < count;
      const uint64_t f = found[inside ? kk : 0];
      const uint32_t off = unit_offset<VEC>(c, v.value_bytes);
      at[b] = inside ? (uint32_t)(f >> kFoundShift) * v.value_bytes + off : kPast;
      const uint8_t* src;
      if constexpr (WHERE == kRowsHbm)
        src = v.values + (uint64_t)(uint32_t)f * v.value_bytes + off;
      else if constexpr (WHERE == kRowsBoth)
        src = value_row(v, inside ? f & kFoundSlot : 0) + off;
      else
        src = inside ? v.host_values + (f & kFoundSlot) * v.value_bytes + off : v.digests;
      buf[b] = load_row_unit<VEC>(src);
      kk += kk_step;
      c += c_step;
      if (c >= units) {
        c -= units;
        kk++;
      }
    }
#pragma unroll
    for (int b = 0; b < kB; b++) store_row_unit<VEC>(dst, at[b], buf[b]);
  }
}

/* Units a lane has in flight: all of a wavefront's for rows of up to 256 bytes (twice as many
 * cost registers: rows of 32 bytes 72 instead of 68 us per 2^20 keys), or a quarter of them where the rows
 * that were found are no more than that: a step past their end costs a load and a store all the same.
 * A row of less than 16 bytes is one or two units. */
template <int VEC, int R, int WHERE>
__device__ __forceinline__ void copy_found_rows(const View& v, const uint64_t* found, uint32_t count,
                                                uint8_t* out, uint64_t base, uint64_t n, int lane) {
  constexpr int kMany = vec_bytes(VEC) == 16 ? 2 * R : (R + 3) / 4;
  constexpr int kFew = kMany / 4 > 1 ? kMany / 4 : 1;
  const uint32_t units = row_units<VEC>(v.value_bytes);
  if (kFew < kMany && units * count <= kWave * kFew)
    copy_units<VEC, R, WHERE, kFew>(v, found, count, units, out, base, n, lane);
  else
    copy_units<VEC, R, WHERE, kMany>(v, found, count, units, out, base, n, lane);
}

/* WAVES wavefronts per workgroup, each with its own keys and its own staging area.  One
 * wavefront per workgroup everywhere except the missed-keys variant, whose workgroups are
 * large so that the list of misses is claimed with one atomic per 1024 keys (updates of one
 * word are served one at a time, about 15 ns each: one per wavefront would take longer than
 * the lookup itself). */
template <int MODE, int VEC, bool DUAL = false, int WAVES = 1, int R = kTile, bool MISSED = false>
__global__ void __launch_bounds__(kWave * WAVES)
lookup_kernel(View v, FindArgs a) {
  __shared__ KeyMeta s_meta_all[WAVES][kWave];
  __shared__ int64_t s_slot_all[WAVES][kWave];
  __shared__ int32_t s_missed[2]; /* misses of the workgroup, start of its part of the list */
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  KeyMeta* const s_meta = s_meta_all[wave];
  int64_t* const s_slot = s_slot_all[wave];
  const uint64_t base = ((uint64_t)blockIdx.x * WAVES + wave) * (kTilesPerWave * R);
  const uint64_t i = lane_owns_key<R>(lane) ? key_of_lane<R>((uint64_t)blockIdx.x * WAVES + wave, lane) : a.n;
  const uint64_t key = stage_keys(v, a.keys, a.n, i, s_meta, s_slot, lane);
  if (DUAL) restage_first_bucket(v, s_meta, lane);
  if (MISSED && threadIdx.x == 0) s_missed[0] = 0;
  wave_sync();
  probe_wave<false, true, R>(v, s_meta, s_slot, nullptr, nullptr, lane);
  wave_sync();
  if (DUAL) {
    restage_second_bucket(v, s_meta, s_slot, lane);
    wave_sync();
    probe_wave<false, true, R>(v, s_meta, s_slot, nullptr, nullptr, lane);
    wave_sync();
  }

  const int64_t my_slot = s_slot[lane];
  if (i < a.n) {
    if (a.founds) a.founds[i] = my_slot >= 0;
    if (my_slot >= 0) {
      if (a.out_scores) a.out_scores[i] = v.scores[my_slot];
      if (MODE == kLookupPtr) a.out_ptrs[i] = value_row(v, (uint64_t)my_slot);
    } else {
      if (MODE == kLookupPtr) a.out_ptrs[i] = nullptr;
    }
  }
  if constexpr (MISSED) {
    /* missed-keys variant (lookup.cuh:36-60): compact list of misses, in no particular
     * order; reserved keys are not probed and count as missed. */
    const bool miss = i < a.n && my_slot < 0;
    const unsigned long long mm = __ballot(miss);
    int32_t at = 0;
    __syncthreads(); /* s_missed has been cleared */
    if (lane == 0 && mm) at = atomicAdd(&s_missed[0], (int32_t)__popcll(mm));
    __syncthreads();
    if (threadIdx.x == 0 && s_missed[0]) s_missed[1] = atomicAdd(a.missed_size, s_missed[0]);
    __syncthreads();
    at = __shfl(at, 0) + s_missed[1];
    if (miss) {
      at += (int32_t)__popcll(mm & ((1ull << lane) - 1));
      a.missed_keys[at] = key;
      a.missed_indices[at] = (int32_t)i;
    }
  }
  if (MODE != kLookupValues) return;

  /* Copy stage: the rows of the keys that were found, spread over the wavefront's 64 lanes.  The keys
   * are listed first, so that a miss costs neither a load nor a store.  All loads of a batch are issued
   * before the first store, and none of them is conditional: a lane past the end of the list reads something
   * all the same (RowsIn), and its store goes past the end of the buffer resource, where the hardware drops
   * it.  Behind a condition every load and store is a block of its own, and the compiler waits for more
   * loads than a store needs.
   * With a step for every key instead of for the found ones, misses cost most of what hits do: 2^20 keys,
   * none found, rows of 256 bytes 50 -> 34 us, of 1024 128 -> 43; half found, rows of 64 bytes 56 -> 49;
   * all found, 256 bytes 103 both ways.  Where at least three quarters of a wavefront's keys are found, the others
   * are listed too: with gaps in the list a store covers parts of lines that the next one completes.  2^19
   * keys, 7/8 found, rows of 512 bytes 90.5 -> 88.8, of 1024 172 -> 168; 2^20 of 400 174 -> 171; rows of 256 bytes and
   * less the same both ways; with the line at half, half found, 400 bytes 110 -> 118. */
  const unsigned long long hits = __ballot(my_slot >= 0);
  if (hits == 0) return;
  constexpr uint32_t kKeys = kTilesPerWave * R;
  const bool most = v.hbm_slots != 0 && (uint32_t)__popcll(hits) * 4 >= kKeys * 3;
  const bool listed = most ? i < a.n : my_slot >= 0;
  const unsigned long long all = __ballot(listed);
  uint64_t* const s_found = reinterpret_cast<uint64_t*>(s_slot); /* every lane has read its slot */
  if (listed)
    s_found[__popcll(all & ((1ull << lane) - 1))] =
        my_slot >= 0 ? (uint64_t)my_slot | ((i - base) << kFoundShift) : kListedMiss;
  wave_sync();
  const uint32_t count = (uint32_t)__popcll(all);
  if (v.hbm_slots >= v.capacity && v.capacity <= 0xFFFFFFFFull)
    copy_found_rows<VEC, R, kRowsHbm>(v, s_found, count, a.out_values, base, a.n, lane);
  else if (v.hbm_slots != 0)
    copy_found_rows<VEC, R, kRowsBoth>(v, s_found, count, a.out_values, base, a.n, lane);
  else
    copy_found_rows<VEC, R, kRowsHost>(v, s_found, count, a.out_values, base, a.n, lane);
}

}  // namespace hkv
#endif
