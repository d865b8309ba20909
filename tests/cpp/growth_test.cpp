/* The bookkeeping that decides whether an inserting call has to sample the load (hkv_growth.hpp), in the orders that
 * several host threads can bring it into.  Prints "all checks passed". */
#include <cstdio>
#include <cstdlib>

#include "hkv_growth.hpp"

using hkv::LoadKnown;

#define CHECK(x)                                                  \
  do {                                                            \
    if (!(x)) {                                                   \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);         \
      std::exit(1);                                               \
    }                                                             \
  } while (0)

static const uint64_t kSlots = 4096;

static uint64_t most(LoadKnown& k, uint64_t n) {
  uint64_t sum = ~UINT64_C(0);
  CHECK(k.most(n, kSlots, sum));
  return sum;
}

static void brings(LoadKnown& k, uint64_t n) { LoadKnown::Call(k, n).enqueue(); }

static void nothing_known() {
  LoadKnown k;
  uint64_t sum = 0;
  LoadKnown::Call mine(k, 5);
  CHECK(!k.most(5, kSlots, sum));
  k.sampled(100, kSlots, 0);
  CHECK(most(k, 5) == 100);
  k.forget();
  CHECK(!k.most(5, kSlots, sum));
  k.sampled(100, kSlots, 0);
  k.recorded();
  CHECK(!k.most(5, kSlots, sum));
}

static void keys_since_the_sample() {
  LoadKnown k;
  for (int call = 0; call < 3; call++) brings(k, 10);
  CHECK(k.enqueued() == 30);
  k.sampled(25, kSlots, k.enqueued());
  for (uint64_t call = 0; call < 4; call++) {
    LoadKnown::Call mine(k, 7);
    CHECK(most(k, 7) == 25 + 7 * call);
    mine.enqueue();
  }
  LoadKnown::Call mine(k, 1), others(k, 6000);
  CHECK(most(k, 1) == kSlots);
}

/* a call is issued; before it asks, another thread issues and enqueues its own and takes a sample that has them */
static void sample_behind_a_later_call() {
  for (uint64_t seen : {0, 3, 50, 1000}) {
    LoadKnown k;
    brings(k, 100);
    LoadKnown::Call mine(k, 10);
    brings(k, 50);
    k.sampled(seen, kSlots, k.enqueued());
    CHECK(most(k, 10) == seen);
    LoadKnown::Call third(k, 20); /* not enqueued: it may come in between */
    CHECK(most(k, 10) == seen + 20);
    third.enqueue();
    CHECK(most(k, 10) == seen + 20);
  }
}

/* a large call that fails before its launches leaves nothing behind, neither for this sample nor for the next */
static void calls_that_fail() {
  LoadKnown k;
  brings(k, 100);
  k.sampled(100, kSlots, k.enqueued());
  for (int call = 0; call < 5; call++) LoadKnown::Call failed(k, 4000);
  LoadKnown::Call mine(k, 10);
  CHECK(most(k, 10) == 100);
  k.sampled(100, kSlots, k.enqueued());
  CHECK(most(k, 10) == 100);
}

/* a sample of another number of slots than the next one would read, which a thread that doubles the table can bring
 * in at any time: half of the slots hold half of the keys */
static void sample_of_other_slots() {
  LoadKnown k;
  uint64_t sum = 0;
  brings(k, 2000);
  k.sampled(1000, kSlots / 2, k.enqueued());
  LoadKnown::Call mine(k, 5);
  CHECK(!k.most(5, kSlots, sum));
  CHECK(k.most(5, kSlots / 2, sum) && sum == 1000);
  k.sampled(2000, kSlots * 2, k.enqueued());
  CHECK(!k.most(5, kSlots, sum));
}

int main() {
  nothing_known();
  keys_since_the_sample();
  sample_behind_a_later_call();
  calls_that_fail();
  sample_of_other_slots();
  std::puts("all checks passed");
}
