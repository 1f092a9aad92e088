// Host checks of csrc/pd_resident.h: prints one line per check that fails.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <chrono>
#include <thread>
#include <vector>

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

// Counts what is held; the allocation number `fail_at` fails, once, after
// its memory was taken when `late` (a device allocation is cleared after it).
struct Alloc {
  int fail_at, late, calls = 0, held = 0;
  template <typename T>
  int device(T** p, size_t n) {
    *p = nullptr;
    const bool fails = calls++ == fail_at;
    if (fails && !late) return 2;
    *p = (T*)malloc(n * sizeof(T));
    ++held;
    return fails ? 2 : 0;
  }
  template <typename T>
  int pinned(T** p) {
    *p = nullptr;
    if (calls++ == fail_at) return 2;
    *p = (T*)malloc(sizeof(T));
    ++held;
    return 0;
  }
  template <typename T>
  void device_free(T*& p) {
    if (p) --held;
    free(p);
    p = nullptr;
  }
  template <typename T>
  void pinned_free(T*& p) {
    device_free(p);
  }
};

static void scratch() {
  for (int late = 0; late < 2; ++late)
    for (int k = -1; k < 4; ++k) {
      Alloc al{k, late};
      pd::SmallScratch s;
      const int first = s.ensure(al, 7, 5);
      CHECK((first != 0) == (k >= 0));
      if (first) {
        CHECK(al.held == 0 && !s.ex && !s.part && !s.aborted && !s.h_aborted);
        CHECK(s.ensure(al, 7, 5) == 0);  // memory is there again
      }
      CHECK(al.held == 4 && s.ex && s.part && s.aborted && s.h_aborted);
      const int calls = al.calls;
      CHECK(s.ensure(al, 7, 5) == 0 && al.calls == calls);
      s.release(al);
      CHECK(al.held == 0 && !s.h_aborted);
    }
}

// `solves` threads of `workgroups` each, two turns apiece: the most at a time.
static int most_at_once(pd::Places& p, int solves, int workgroups) {
  const int k = pd::Places::needed(workgroups, 8);
  std::atomic<int> now{0}, most{0};
  std::vector<std::thread> t;
  for (int i = 0; i < solves; ++i)
    t.emplace_back([&] {
      for (int turn = 0; turn < 2; ++turn) {
        pd::PlacesHeld held(p, k);
        const int mine = ++now;
        for (int m = most; mine > m && !most.compare_exchange_weak(m, mine);) {
        }
        std::this_thread::sleep_for(std::chrono::milliseconds(20));
        --now;
      }
    });
  for (auto& th : t) th.join();
  return most;
}

static void places() {
  CHECK(pd::Places::needed(1, 8) == 1 && pd::Places::needed(8, 8) == 1);
  CHECK(pd::Places::needed(20, 8) == 3 && pd::Places::needed(256, 8) == 32);
  pd::Places p(32);
  CHECK(most_at_once(p, 16, 20) == 10);   // 288 rows: 3 places each
  CHECK(most_at_once(p, 5, 128) == 2);
  CHECK(most_at_once(p, 5, 129) == 1);    // 17 + 17 > 32
  CHECK(most_at_once(p, 3, 256) == 1);
  // a solve of the whole device comes to its turn among small ones
  std::atomic<bool> stop{false};
  std::vector<std::thread> small;
  for (int i = 0; i < 4; ++i)
    small.emplace_back([&] {
      while (!stop) {
        pd::PlacesHeld held(p, 3);
        std::this_thread::sleep_for(std::chrono::milliseconds(1));
      }
    });
  std::this_thread::sleep_for(std::chrono::milliseconds(5));
  { pd::PlacesHeld held(p, 32); }
  stop = true;
  for (auto& th : small) th.join();
  p.take(32);  // everything was given back
  p.give(32);
}

int main(int argc, char** argv) {
  if (argc > 1 && !strcmp(argv[1], "wait_limit")) wait_limit();
  else if (argc > 1 && !strcmp(argv[1], "scratch")) scratch();
  else if (argc > 1 && !strcmp(argv[1], "places")) places();
  else return 2;
  return bad ? 1 : 0;
}
