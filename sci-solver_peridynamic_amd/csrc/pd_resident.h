// pd_resident.h -- the rules of the resident solve (pd_small.hip) that need no
// device: plain C++, also compiled by the tests for the host.
#pragma once

#include <condition_variable>
#include <cstddef>
#include <deque>
#include <mutex>

#if defined(__HIPCC__)
#define PD_HD __host__ __device__ __forceinline__
#else
#define PD_HD inline
#endif

namespace pd {

// The limit of one wait, in ticks.  The clock is read on every 16th poll only
// (a wait of an undisturbed solve takes a microsecond or two and fewer polls
// than that), and counts from the first reading of this wait: a solve may
// last as long as it makes progress.
struct WaitLimit {
  unsigned long long limit;
  unsigned long long since = 0;
  PD_HD explicit WaitLimit(unsigned long long ticks) : limit(ticks) {}
  PD_HD static bool due(unsigned poll) { return (poll & 15) == 15; }
  PD_HD bool over(unsigned poll, unsigned long long now) {
    if (poll == 15) since = now;
    return now - since > limit;
  }
};

// Room for resident solves on a device, shared by its contexts: all workgroups
// of a solve must find a CU while those of other solves wait in theirs, so a
// solve takes its places ahead of its launch and gives them back when it has
// finished.  Workgroups are dealt to the XCDs in turn, so a solve of u
// workgroups needs at most ceil(u / xcds) CUs on any of them, and that is what
// is counted: counting CUs of the whole device would let solves whose
// remainders fall on the same XCD hold each other up there.
//
// Who finds room goes ahead of those who wait, up to kPasses times in a row,
// then the first in line is next: handing the places to a sleeping thread
// leaves the device idle until it has woken (13k rows, a solve of which fills
// the device, 12 threads: 3.8 thousand steps a second in strict order, 4.3
// so, as with a lock), and a solve that needs the whole device still comes to
// its turn.  288 rows, 8 threads: 10.3 thousand steps a second with one solve
// at a time, 40.4 side by side.
class Places {
 public:
  explicit Places(int total = 0) : total_(total) {}
  static int needed(int workgroups, int xcds) { return (workgroups + xcds - 1) / xcds; }
  void take(int k) {
    std::unique_lock<std::mutex> lock(mu_);
    if (used_ + k <= total_ && (line_.empty() || passes_ < kPasses)) {
      if (!line_.empty()) ++passes_;
      used_ += k;
      return;
    }
    std::condition_variable mine;
    line_.push_back(&mine);
    mine.wait(lock, [&] { return line_.front() == &mine && used_ + k <= total_; });
    line_.pop_front();
    passes_ = 0;
    used_ += k;
    if (!line_.empty()) line_.front()->notify_one();  // there may be room for it too
  }
  void give(int k) {
    std::lock_guard<std::mutex> lock(mu_);
    used_ -= k;
    if (!line_.empty()) line_.front()->notify_one();
  }

 private:
  static constexpr int kPasses = 16;
  std::mutex mu_;
  std::deque<std::condition_variable*> line_;  // the waiting, each on its own stack
  const int total_;
  int used_ = 0, passes_ = 0;
};

// Places held for as long as this lives.
class PlacesHeld {
 public:
  PlacesHeld(Places& p, int k) : p_(p), k_(k) { p_.take(k_); }
  ~PlacesHeld() { p_.give(k_); }
  PlacesHeld(const PlacesHeld&) = delete;
  PlacesHeld& operator=(const PlacesHeld&) = delete;

 private:
  Places& p_;
  const int k_;
};

// A context's scratch for the resident step, there as a whole or not at all:
// a step that could not allocate it reports that, and so does the next one.
// Alloc: int device(T**, count), int pinned(T**), 0 on success, and
// device_free(T*&), pinned_free(T*&), which take null.
struct SmallScratch {
  double* ex = nullptr;               // [2][n][6]
  double* part = nullptr;             // [9][row]
  unsigned int* aborted = nullptr;    // device word
  unsigned int* h_aborted = nullptr;  // pinned
  template <class Alloc>
  int ensure(Alloc& al, size_t n, size_t row) {
    if (h_aborted) return 0;  // allocated last
    int e;
    if ((e = al.device(&ex, 12 * n)) || (e = al.device(&part, 9 * row)) ||
        (e = al.device(&aborted, 1)) || (e = al.pinned(&h_aborted)))
      release(al);
    return e;
  }
  template <class Alloc>
  void release(Alloc& al) {
    al.device_free(ex);
    al.device_free(part);
    al.device_free(aborted);
    al.pinned_free(h_aborted);
  }
};

}  // namespace pd
