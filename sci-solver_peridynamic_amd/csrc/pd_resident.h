// pd_resident.h -- the rules of the resident solve (pd_small.hip) that need no
// device: plain C++, also compiled by the tests for the host.
#pragma once

#include <cstddef>

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
