// pd_resident.h -- the rules of the resident solve (pd_small.hip) that need no
// device: plain C++, also compiled by the tests for the host.
#pragma once

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

}  // namespace pd
