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

static int launches = 0, fail_launch = -1; /* of the launches from now on, the one that fails */
static hipError_t last = hipSuccess;

extern "C" {
hipError_t hipMallocAsync(void** p, size_t bytes, hipStream_t) {
  *p = std::malloc(bytes);
  return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) {
  std::free(p);
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

int main() {
  failed_launches();
  numbers_of_calls();
  std::puts("all checks passed");
}
