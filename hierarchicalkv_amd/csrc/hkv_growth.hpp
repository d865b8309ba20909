/*
 * What the host knows about the load of a table that can grow: the last load sample and the keys that have been handed
 * to upserts since.  No HIP here.
 */
#ifndef HKV_GROWTH_HPP_
#define HKV_GROWTH_HPP_

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <mutex>

namespace hkv {

class LoadKnown {
 public:
  /* The keys of one call: issued when it begins, before anything else of it is done, enqueued when its kernels are
   * about to be launched and the call has the table to itself (inserter role of the group lock).  A call that returns
   * before that, with an error, brings none: they are taken back. */
  class Call {
   public:
    Call(LoadKnown& k, uint64_t n) : k_(k), n_(n), open_(true) { k_.issued_ += n_; }
    Call(const Call&) = delete;
    Call& operator=(const Call&) = delete;
    ~Call() {
      if (open_) k_.issued_ -= n_;
    }
    void enqueue() {
      k_.enqueued_ += n_;
      open_ = false;
    }

   private:
    LoadKnown& k_;
    const uint64_t n_;
    bool open_;
  };
  uint64_t enqueued() const { return enqueued_; }

  /* a sample of `slots` slots that ran behind the first `at` enqueued keys read `sum` */
  void sampled(uint64_t sum, uint64_t slots, uint64_t at) {
    std::lock_guard<std::mutex> g(mu_);
    sum_ = sum;
    slots_ = slots;
    at_ = at;
  }
  void forget() { sampled(0, 0, 0); }
  /* upserts have been recorded into a graph: nobody counts what its replays bring */
  void recorded() { untracked_ = true; }

  /* The most that a sample of `slots` slots could read now, for a call of n keys that has been issued and not been
   * enqueued; false where nothing is known of that many slots (another thread may have doubled a small table, of which
   * the next sample reads more).  Every key enqueued behind the sample may have come into its slots, and the keys of calls that other
   * threads are about to enqueue may have as well.  Each enqueued key was issued before and this call's are not
   * enqueued, so what is issued without them is never below what the sample has seen, whichever thread took it. */
  bool most(uint64_t n, uint64_t slots, uint64_t& sum) {
    if (untracked_) return false;
    std::lock_guard<std::mutex> g(mu_);
    if (slots_ != slots) return false;
    sum = std::min(slots, sum_ + (issued_ - n - at_));
    return true;
  }

 private:
  std::atomic<uint64_t> issued_{0};   /* keys handed to upserts since creation */
  std::atomic<uint64_t> enqueued_{0}; /* the same, of calls that came to their launches */
  std::mutex mu_;
  uint64_t sum_ = 0;
  uint64_t slots_ = 0; /* 0: nothing is known */
  uint64_t at_ = 0;
  std::atomic<bool> untracked_{false};
};

}  // namespace hkv
#endif
