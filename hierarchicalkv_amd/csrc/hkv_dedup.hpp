/*
 * Batches that may hold a key more than once (unique_key = false).
 *
 * The reference switches to its lock-per-bucket kernels for such batches
 * (merlin_hashtable.cuh:1194-1252, 1737-1790, 1925-1960): every occurrence is applied,
 * in no particular order, and the table ends up holding the key once (tests/
 * find_or_insert_ptr_test.cc.cu:3390-3475: 1024 copies of one key leave one entry).  Here
 * the batch is reduced to one occurrence per key: the first
 * occurrence stands for the key, and the upsert takes the others for the EMPTY key, which
 * every kernel skips.  Calls that hand something back per key (find_or_insert) copy it from
 * the representative afterwards.
 *
 * The first occurrences are found with an open-addressing index of the batch.  A workgroup
 * settles the repetitions among its own keys in LDS and brings one entry per key to the index in
 * device memory, so that a key that makes up a fifteenth of a batch (ids of a recommender are
 * Zipf-distributed) costs one atomic per workgroup and not one per occurrence: atomics on one word
 * are served one at a time, about 15 ns each.  An entry is a word of 16 hash bits, the number of the call and the index of
 * the lowest occurrence seen so far: a minimum on the word keeps the lowest one, and keys are only
 * fetched for comparison where the hash bits agree.  An entry of another call counts as free, so that the index, which a
 * table keeps, is cleared once in 65 535 calls, and the upsert looks up for itself whether a key stands for the others
 * of its kind: a launch of its own takes 4 us however little it does.  What is left is bound by one 8-byte atomic on a random
 * line per distinct key of a workgroup and by the queue at the most frequent keys.
 * 2^18 keys of 32 floats, Zipf(1.05) over 2^21 ids, the whole find_or_insert + insert_or_assign: 129 us with a clear
 * before and a pass over the keys behind every call's index (3.5 and 4.5 us), 116 without, 114 as it is here.
 */
#ifndef HKV_DEDUP_HPP_
#define HKV_DEDUP_HPP_

#include "hkv_common.hpp"

namespace hkv {

/* entries that no call has made */
constexpr uint32_t kNoCall = 0xFFFF;

__global__ void __launch_bounds__(256)
dedup_clear_kernel(uint64_t* index, uint64_t words) {
  const uint64_t q = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 2;
  if (q < words) *reinterpret_cast<uint4*>(index + q) = make_uint4(~0u, ~0u, ~0u, ~0u);
}

/* Enters every key of the batch; at[i] = the place in the index of key i's entry.  `mask` + 1
 * entries, at least twice as many as keys, so that a free one always ends the search; two neighbours, which one load brings,
 * are tried before the next pair.  One key per
 * thread: two or four of them meant fewer, longer workgroups and were slower at every size. */
template <int THREADS>
__global__ void __launch_bounds__(THREADS)
dedup_enter_kernel(const uint64_t* keys, uint64_t n, uint64_t* index, uint64_t mask, uint32_t call, uint32_t* at) {
  constexpr uint32_t kPlaces = 2 * THREADS; /* half of them stay free */
  __shared__ uint64_t s_key[THREADS];
  __shared__ uint32_t s_index[kPlaces]; /* lowest thread with the key, ~0: free */
  __shared__ uint32_t s_at[THREADS];    /* of that thread's key: where its entry is */
  const uint32_t l = threadIdx.x;
  const uint64_t i = (uint64_t)blockIdx.x * THREADS + l;
  const bool valid = i < n;
  const uint64_t key = valid ? keys[i] : 0;
  const uint64_t h = fmix64(key);
  /* the place and the hash bits of the entry have no bit in common below 2^31 keys (2^47 entries) */
  uint64_t where = (h >> 16) & mask;
  const uint64_t mine = (h << 48) | ((uint64_t)call << 32) | i;
  /* How the places look now: an entry of this call stays where it is once it is there, so whatever stands
   * there needs no atomic.  The load is under way while the workgroup sorts out its own keys. */
  uint4 pair = *reinterpret_cast<const uint4*>(index + (where & ~UINT64_C(1)));
  s_key[l] = key;
  s_index[l] = s_index[l + THREADS] = ~0u;
  __syncthreads();
  uint32_t place = (uint32_t)h & (kPlaces - 1);
  while (valid) {
    const uint32_t old = atomicCAS(&s_index[place], ~0u, l);
    if (old == ~0u) break;
    if (s_key[old] == key) { /* whichever of the key's threads stands there */
      if (l < old) atomicMin(&s_index[place], l);
      break;
    }
    place = (place + 1) & (kPlaces - 1);
  }
  __syncthreads();
  if (valid && s_index[place] == l) {
    unsigned long long* const words = reinterpret_cast<unsigned long long*>(index);
    for (uint32_t tried = 1;; tried++) {
      unsigned long long old = (where & 1) ? (pair.z | ((unsigned long long)pair.w << 32)) : (pair.x | ((unsigned long long)pair.y << 32));
      if ((uint32_t)(old >> 32 & 0xFFFF) != call) {
        const unsigned long long stale = old;
        old = atomicCAS(words + where, stale, (unsigned long long)mine);
        if (old == stale) break;
      }
      if ((old >> 32) == (mine >> 32) && keys[(uint32_t)old] == key) {
        if (i < (uint32_t)old) atomicMin(words + where, (unsigned long long)mine);
        break;
      }
      where ^= 1;
      if ((tried & 1) == 0) {
        where = ((where | 1) + 1) & mask;
        pair = *reinterpret_cast<const uint4*>(index + where);
      }
    }
    s_at[l] = (uint32_t)where;
  }
  __syncthreads();
  if (valid) at[i] = s_at[s_index[place]];
}

/* what a duplicate gets back: the representative's pointer and flag ... */
__global__ void dedup_fix_ptrs_kernel(const uint32_t* rep, uint64_t n, void** out_ptrs, uint8_t* founds) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t r = rep[i];
  if (r == (uint32_t)i) return;
  if (out_ptrs) out_ptrs[i] = out_ptrs[r];
  if (founds) founds[i] = founds[r];
}
/* ... or its row, one T per thread: keys first .. first + n - 1.  The rows that are read belong to
 * representatives, which nobody writes.  2^18 rows of 128 bytes, Zipf(1.05): 6 us; 59 us with a workgroup per
 * key, 18 us with four copies in flight per thread or with a list of the duplicates per wavefront. */
template <class T>
__global__ void __launch_bounds__(256)
dedup_fix_rows_kernel(const uint32_t* rep, uint64_t first, uint32_t n, uint8_t* rows, uint32_t row_bytes) {
  const uint32_t units = row_bytes / sizeof(T);
  const uint32_t u = blockIdx.x * 256u + threadIdx.x;
  if (u >= n * units) return;
  const uint64_t i = first + u / units;
  const uint32_t r = rep[i];
  if (r == (uint32_t)i) return;
  const uint32_t c = u % units;
  reinterpret_cast<T*>(rows + i * row_bytes)[c] = reinterpret_cast<const T*>(rows + r * (uint64_t)row_bytes)[c];
}

/* (4 GiB of rows are a possible batch on this card; a row is at most 2^20 bytes) */
template <class T>
inline void dedup_fix_rows_by(const uint32_t* rep, uint64_t n, uint8_t* rows, uint32_t row_bytes, hipStream_t s) {
  const uint64_t units = row_bytes / sizeof(T), step = kLaunchThreads / units;
  for (uint64_t first = 0; first < n; first += step) {
    const uint64_t m = n - first < step ? n - first : step;
    hipLaunchKernelGGL(dedup_fix_rows_kernel<T>, dim3((unsigned)((m * units + 255) / 256)), dim3(256), 0, s, rep, first,
                       (uint32_t)m, rows, row_bytes);
  }
}
inline void dedup_fix_rows(const uint32_t* rep, uint64_t n, uint8_t* rows, uint32_t row_bytes, hipStream_t s) {
  const uintptr_t mis = row_bytes | (uintptr_t)rows;
  if ((mis & 15) == 0)
    dedup_fix_rows_by<uint4>(rep, n, rows, row_bytes, s);
  else if ((mis & 3) == 0)
    dedup_fix_rows_by<uint32_t>(rep, n, rows, row_bytes, s);
  else
    dedup_fix_rows_by<uint8_t>(rep, n, rows, row_bytes, s);
}

/* The index of a batch: memory for `keys` keys, `sparse` entries per key at least, and the number of the last call that
 * used it.  Four entries per key instead of two shorten the longest search of a workgroup, which all its keys wait for:
 * find_or_insert + insert_or_assign of Zipf-distributed ids, 70 000 of 128 bytes 60.9 -> 59.4 us, 2^17 of 64 bytes
 * 73.4 -> 71.0, 2^18 of 128 bytes 111.7 -> 109.9, 500 000 the same.  An index that goes with the call is cleared by
 * it and takes two. */
struct RepeatIndex {
  uint8_t* block = nullptr;
  uint64_t keys = 0;
  uint32_t sparse = 2;
  uint32_t call = 0;
};
inline uint64_t repeat_entries(uint64_t keys, uint32_t sparse) {
  uint64_t entries = 64;
  while (entries < sparse * keys) entries *= 2;
  return entries;
}
/* Where an index comes from and goes back to, in the order of the stream */
struct StreamMemory {
  static hipError_t take(void** p, size_t bytes, hipStream_t s) { return hipMallocAsync(p, bytes, s); }
  static void give(void* p, hipStream_t s) { (void)hipFreeAsync(p, s); }
};
template <class Memory>
hipError_t repeat_index_make(RepeatIndex& x, uint64_t keys, uint32_t sparse, Memory memory, hipStream_t s) {
  const uint64_t entries = repeat_entries(keys, sparse);
  const hipError_t e = memory.take((void**)&x.block, entries * 8 + keys * 4, s);
  if (e != hipSuccess) {
    x.block = nullptr;
    return e;
  }
  x.keys = keys;
  x.sparse = sparse;
  x.call = kNoCall; /* to be cleared */
  return hipSuccess;
}
template <class Memory>
void repeat_index_free(RepeatIndex& x, Memory memory, hipStream_t s) {
  if (x.block) memory.give(x.block, s);
  x = RepeatIndex{};
}

/* The index for a batch of n keys: the table's own, `kept`, made large enough, for batches of up to `most_kept` keys;
 * for others, and where that much memory is not to be had, one that goes with the call and takes less, `own`. */
template <class Memory>
hipError_t repeat_index_for(uint64_t n, uint64_t most_kept, RepeatIndex& kept, Memory memory, RepeatIndex& own, hipStream_t s,
                            RepeatIndex*& x) {
  x = &kept;
  if (n <= most_kept) {
    if (kept.keys >= n) return hipSuccess;
    repeat_index_free(kept, memory, s);
    uint64_t keys = UINT64_C(1) << 12;
    while (keys < n) keys *= 2;
    if (keys > most_kept) keys = most_kept;
    if (repeat_index_make(kept, keys, 4, memory, s) == hipSuccess) return hipSuccess;
    (void)hipGetLastError();
  }
  x = &own;
  return repeat_index_make(own, n, 2, StreamMemory(), s);
}

/* Enters the n keys of a batch (n < 2^31, at most x.keys) on stream s; the upsert gets `index` and `rep`.  Where a launch
 * fails nobody knows what is in the index: the next call that uses it clears it. */
inline hipError_t repeat_index_enter(RepeatIndex& x, uint64_t n, const uint64_t* keys, hipStream_t s, const uint64_t*& index_out,
                               uint32_t*& rep) {
  const uint64_t all = repeat_entries(x.keys, x.sparse), entries = repeat_entries(n, x.sparse);
  uint64_t* const index = (uint64_t*)x.block;
  rep = (uint32_t*)(x.block + all * 8);
  index_out = index;
  if (++x.call >= kNoCall) {
    hipLaunchKernelGGL(dedup_clear_kernel, dim3((unsigned)((all / 2 + 255) / 256)), dim3(256), 0, s, index, all);
    x.call = 0;
  }
  /* Large workgroups keep the queues at the frequent keys short (2^20 keys: 48 us with 1024 threads,
   * 90 with 256), small ones get more CUs to work on a small batch (2^12 keys: 4 and 7 us; the
   * lines cross between 2^15 and 2^16). */
  if (n >= (UINT64_C(1) << 15))
    hipLaunchKernelGGL(dedup_enter_kernel<1024>, dim3((unsigned)((n + 1023) / 1024)), dim3(1024), 0, s, keys, n, index,
                       entries - 1, x.call, rep);
  else
    hipLaunchKernelGGL(dedup_enter_kernel<256>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, keys, n, index,
                       entries - 1, x.call, rep);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) x.call = kNoCall;
  return e;
}

}  // namespace hkv
#endif
