/*
 * Batches that may hold a key more than once (unique_key = false).
 *
 * The reference switches to its lock-per-bucket kernels for such batches
 * (merlin_hashtable.cuh:1194-1252, 1737-1790, 1925-1960): every occurrence is applied,
 * in no particular order, and the table ends up holding the key once (tests/
 * find_or_insert_ptr_test.cc.cu:3390-3475: 1024 copies of one key leave one entry).  Here
 * the batch is reduced to one occurrence per key before the ordinary kernels run: the first
 * occurrence stands for the key, and the other occurrences travel as the EMPTY key, which
 * every kernel skips.  Calls that hand something back per key (find_or_insert) copy it from
 * the representative afterwards.
 *
 * The first occurrences are found with an open-addressing index of the batch.  A workgroup
 * settles the repetitions among its own keys in LDS and brings one entry per key to the index in
 * device memory, so that a key that makes up a fifteenth of a batch (ids of a recommender are
 * Zipf-distributed) costs one atomic per workgroup and not one per occurrence: atomics on one word
 * are served one at a time, about 15 ns each.  An entry is a word of 32 hash bits and the index of
 * the lowest occurrence seen so far: a minimum on the word keeps the lowest one, and keys are only
 * fetched for comparison where the hash bits agree.  It is bound by one 8-byte atomic on a random
 * line per distinct key of a workgroup and by the queue at the most frequent keys.
 * 2^18 keys of 32 floats, Zipf(1.05) over 2^21 ids, the whole find_or_insert + insert_or_assign:
 * 0.383 ms with a radix sort of (key, index) and a running maximum (18 launches, 0.125 ms a batch),
 * 0.13 ms as it is here (clear 4, enter 18, mark 5 us).
 */
#ifndef HKV_DEDUP_HPP_
#define HKV_DEDUP_HPP_

#include "hkv_common.hpp"

namespace hkv {

struct DedupPlan {
  uint64_t* keys = nullptr; /* [n] the batch with later occurrences replaced by EMPTY */
  uint32_t* rep = nullptr;  /* [n] index of the occurrence that stands for key i */
  void* block = nullptr;
  hipStream_t stream = nullptr;
};

constexpr uint64_t kDedupFree = UINT64_C(0xFFFFFFFFFFFFFFFF);

__global__ void __launch_bounds__(256)
dedup_clear_kernel(uint64_t* index, uint64_t words) {
  const uint64_t q = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 2;
  if (q < words) *reinterpret_cast<uint4*>(index + q) = make_uint4(~0u, ~0u, ~0u, ~0u);
}

/* Enters every key of the batch; at[i] = the place in the index of key i's entry.  `mask` + 1
 * entries, at least twice as many as keys, so that a free one always ends the search.  One key per
 * thread: two or four of them meant fewer, longer workgroups and were slower at every size. */
template <int THREADS>
__global__ void __launch_bounds__(THREADS)
dedup_enter_kernel(const uint64_t* keys, uint64_t n, uint64_t* index, uint64_t mask, uint32_t* at) {
  constexpr uint32_t kPlaces = 2 * THREADS; /* half of them stay free */
  __shared__ uint64_t s_key[THREADS];
  __shared__ uint32_t s_index[kPlaces]; /* lowest thread with the key, ~0: free */
  __shared__ uint32_t s_at[THREADS];    /* of that thread's key: where its entry is */
  const uint32_t l = threadIdx.x;
  const uint64_t i = (uint64_t)blockIdx.x * THREADS + l;
  const bool valid = i < n;
  const uint64_t key = valid ? keys[i] : 0;
  const uint64_t h = fmix64(key);
  /* the place and the hash bits of the entry have no bit in common below 2^31 keys */
  uint64_t where = (h >> 32) & mask;
  const uint64_t mine = (h << 32) | i;
  /* How the place looks now: an entry stays where it is once it is there, so whatever stands
   * there needs no atomic.  The load is under way while the workgroup sorts out its own keys. */
  unsigned long long ahead = index[where];
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
    for (;;) {
      const unsigned long long old =
          ahead != kDedupFree ? ahead : atomicCAS(words + where, (unsigned long long)kDedupFree, (unsigned long long)mine);
      ahead = kDedupFree;
      if (old == kDedupFree) break;
      if ((uint32_t)(old >> 32) == (uint32_t)h && keys[(uint32_t)old] == key) {
        if (i < (uint32_t)old) atomicMin(words + where, (unsigned long long)mine);
        break;
      }
      where = (where + 1) & mask;
    }
    s_at[l] = (uint32_t)where;
  }
  __syncthreads();
  if (valid) at[i] = s_at[s_index[place]];
}

/* `rep` comes in as the place of every key's entry and becomes the occurrence that stands for it */
__global__ void __launch_bounds__(256)
dedup_mark_kernel(const uint64_t* keys, uint64_t n, const uint64_t* index, uint64_t empty_key, uint64_t* keys_mod,
                  uint32_t* rep) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t first = (uint32_t)index[rep[i]];
  rep[i] = first;
  keys_mod[i] = first == (uint32_t)i ? keys[i] : empty_key;
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

inline void dedup_free(DedupPlan& d) {
  if (d.block) (void)hipFreeAsync(d.block, d.stream);
  d.block = nullptr;
}

/* Builds d.keys and d.rep for the n keys of a batch on stream s (n < 2^31). */
inline hipError_t dedup_make(const View& v, uint64_t n, const uint64_t* keys, hipStream_t s,
                             DedupPlan& d) {
  d.stream = s;
  auto up = [](uint64_t x) { return (x + 255) & ~UINT64_C(255); };
  uint64_t entries = 64;
  while (entries < 2 * n) entries *= 2;
  const uint64_t o_rep = up(n * 8);
  const uint64_t o_index = o_rep + up(n * 4);
  hipError_t e = hipMallocAsync(&d.block, o_index + entries * 8, s);
  if (e != hipSuccess) return e;
  uint8_t* b = (uint8_t*)d.block;
  d.keys = (uint64_t*)b;
  d.rep = (uint32_t*)(b + o_rep);
  uint64_t* index = (uint64_t*)(b + o_index);
  hipLaunchKernelGGL(dedup_clear_kernel, dim3((unsigned)((entries / 2 + 255) / 256)), dim3(256), 0, s, index, entries);
  /* Large workgroups keep the queues at the frequent keys short (2^20 keys: 48 us with 1024 threads,
   * 90 with 256), small ones get more CUs to work on a small batch (2^12 keys: 4 and 7 us; the
   * lines cross between 2^15 and 2^16). */
  if (n >= (UINT64_C(1) << 15))
    hipLaunchKernelGGL(dedup_enter_kernel<1024>, dim3((unsigned)((n + 1023) / 1024)), dim3(1024), 0, s, keys, n, index,
                       entries - 1, d.rep);
  else
    hipLaunchKernelGGL(dedup_enter_kernel<256>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, keys, n, index,
                       entries - 1, d.rep);
  hipLaunchKernelGGL(dedup_mark_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, keys, n,
                     (const uint64_t*)index, v.empty_key, d.keys, d.rep);
  e = hipGetLastError();
  if (e != hipSuccess) dedup_free(d);
  return e;
}

}  // namespace hkv
#endif
