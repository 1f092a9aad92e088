// Host checks of csrc/pd_resident.h: prints one line per check that fails.
#include <cstdio>
#include <cstring>

#include "pd_resident.h"

static int bad = 0;
#define CHECK(c) \
  do { \
    if (!(c)) { \
      ++bad; \
      printf("%s:%d: %s\n", __FILE__, __LINE__, #c); \
    } \
  } while (0)

// One wait of `polls` polls, 70 ticks each, from *clock on; whether it was given up.
static bool wait(unsigned long long limit, unsigned polls, unsigned long long* clock) {
  pd::WaitLimit w(limit);
  for (unsigned k = 0; k < polls; ++k) {
    *clock += 70;
    if (pd::WaitLimit::due(k) && w.over(k, *clock)) return true;
  }
  return false;
}

static void wait_limit() {
  unsigned long long clock = 1ull << 40;
  const unsigned long long start = clock, limit = 100000;
  // every wait reads the clock, none lasts for long, all together for 1000 limits
  bool up = false;
  for (int k = 0; k < 40000; ++k) up = up || wait(limit, 40, &clock);
  CHECK(!up);
  CHECK(clock - start > 1000 * limit);
  // one wait past the limit ends, soon after it
  const unsigned long long before = clock;
  CHECK(wait(limit, 1u << 30, &clock));
  CHECK(clock - before > limit && clock - before < limit + 40 * 70);
  // one below it does not
  CHECK(!wait(limit, 1400, &clock));
}

int main(int argc, char** argv) {
  if (argc > 1 && !strcmp(argv[1], "wait_limit")) wait_limit();
  else return 2;
  return bad ? 1 : 0;
}
