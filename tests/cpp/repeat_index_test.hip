/* The host side of the index of repeated keys (hkv_dedup.hpp) where HIP calls fail.  The calls it makes are defined here, so
 * that nothing reaches a GPU: memory is the host's, a launch is counted and may be told to fail.
 * Prints "all checks passed". */
#include <cstdio>
#include <cstdlib>

#include "hkv_dedup.hpp"

#define CHECK(x)                                          \
  do {                                                    \
    if (!(x)) {                                           \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x); \
      std::exit(1);                                       \
    }                                                     \
  } while (0)

static size_t largest = ~size_t(0), taken = 0; /* block that is to be had; bytes of the last one */
static int blocks = 0;
static int launches = 0, fail_launch = -1; /* of the launches from now on, the one that fails */
static hipError_t last = hipSuccess;

extern "C" {
hipError_t hipMallocAsync(void** p, size_t bytes, hipStream_t) {
  if (bytes > largest) return last = hipErrorOutOfMemory;
  *p = std::malloc(taken = bytes);
  blocks++;
  return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) {
  std::free(p);
  blocks--;
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
  launches++;
  if (fail_launch-- == 0) last = hipErrorLaunchFailure;
  return last;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
}

using namespace hkv;

static int enter(RepeatIndex& x, uint64_t n, hipError_t want) {
  const uint64_t* index = nullptr;
  uint32_t* rep = nullptr;
  launches = 0;
  CHECK(repeat_index_enter(x, n, nullptr, nullptr, index, rep) == want);
  return launches;
}

static void failed_launches() {
  for (uint64_t n : {100, 40000}) {
    RepeatIndex x;
    CHECK(repeat_index_make(x, 40000, 4, StreamMemory(), nullptr) == hipSuccess);
    fail_launch = 0; /* the clear */
    enter(x, n, hipErrorLaunchFailure);
    CHECK(enter(x, n, hipSuccess) == 2); /* clears again */
    CHECK(enter(x, n, hipSuccess) == 1);
    fail_launch = 0; /* the keys */
    CHECK(enter(x, n, hipErrorLaunchFailure) == 1);
    fail_launch = 1; /* ... behind a clear */
    CHECK(enter(x, n, hipErrorLaunchFailure) == 2);
    CHECK(enter(x, n, hipSuccess) == 2);
    CHECK(enter(x, n, hipSuccess) == 1);
    repeat_index_free(x, StreamMemory(), nullptr);
  }
}

static void numbers_of_calls() {
  RepeatIndex x;
  CHECK(repeat_index_make(x, 64, 4, StreamMemory(), nullptr) == hipSuccess);
  for (int round = 0; round < 2; round++) {
    CHECK(enter(x, 64, hipSuccess) == 2 && x.call == 0);
    for (uint32_t call = 1; call < kNoCall; call++) CHECK(enter(x, 64, hipSuccess) == 1 && x.call == call);
  }
  repeat_index_free(x, StreamMemory(), nullptr);
}

static RepeatIndex* index_for(uint64_t n, uint64_t most_kept, RepeatIndex& kept, RepeatIndex& own) {
  RepeatIndex* x = nullptr;
  CHECK(repeat_index_for(n, most_kept, kept, StreamMemory(), own, nullptr, x) == hipSuccess);
  CHECK(x->keys >= n && (x == &kept || x == &own));
  CHECK(enter(*x, n, hipSuccess) >= 1);
  return x;
}

static void kept_or_not() {
  RepeatIndex kept, own;
  const uint64_t most = 1 << 16;
  CHECK(index_for(10, most, kept, own) == &kept && blocks == 1 && kept.keys == 4096);
  CHECK(index_for(4096, most, kept, own) == &kept && blocks == 1 && kept.keys == 4096);
  CHECK(index_for(4097, most, kept, own) == &kept && blocks == 1 && kept.keys == 8192);
  CHECK(index_for(most, most, kept, own) == &kept && blocks == 1 && kept.keys == most);
  CHECK(index_for(5, most, kept, own) == &kept && kept.keys == most && kept.call == 1);
  CHECK(index_for(most + 1, most, kept, own) == &own && blocks == 2 && own.sparse == 2);
  repeat_index_free(own, StreamMemory(), nullptr);
  CHECK(index_for(5, 0, kept, own) == &own && blocks == 2);
  repeat_index_free(own, StreamMemory(), nullptr);
  repeat_index_free(kept, StreamMemory(), nullptr);
  CHECK(index_for(10, 384, kept, own) == &kept && kept.keys == 384); /* no more than may be kept */
  CHECK(index_for(385, 384, kept, own) == &own);
  repeat_index_free(own, StreamMemory(), nullptr);
  repeat_index_free(kept, StreamMemory(), nullptr);
  CHECK(blocks == 0);
}

/* memory for an index of four entries per key is not to be had, for two it is: the call goes on with that, and with an index that is
 * kept once there is memory again; with none the call fails and says so */
static void memory_runs_out() {
  RepeatIndex kept, own;
  const uint64_t n = 1 << 15, most = 1 << 16;
  CHECK(index_for(100, most, kept, own) == &kept);
  largest = n * 28;
  CHECK(index_for(n, most, kept, own) == &own && own.sparse == 2 && taken <= largest && !kept.block && blocks == 1);
  CHECK(last == hipSuccess);
  repeat_index_free(own, StreamMemory(), nullptr);
  CHECK(index_for(100, most, kept, own) == &kept);
  largest = 100;
  RepeatIndex* x = nullptr;
  CHECK(repeat_index_for(n, most, kept, StreamMemory(), own, nullptr, x) == hipErrorOutOfMemory && !own.block);
  last = hipSuccess;
  largest = ~size_t(0);
  CHECK(index_for(n, most, kept, own) == &kept);
  repeat_index_free(own, StreamMemory(), nullptr);
  repeat_index_free(kept, StreamMemory(), nullptr);
  CHECK(blocks == 0);
}

int main() {
  failed_launches();
  kept_or_not();
  memory_runs_out();
  numbers_of_calls();
  std::puts("all checks passed");
}
