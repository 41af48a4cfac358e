// Host-side checks of the persistent PCG's index and epoch rules
// (hip/pcg_rules.hpp) and exchange memory (hip/pcg_words.hpp), and of the CCD
// search's re-reads of the minimum (hip/ccd_rules.hpp).
// Prints the first failure and returns 1; run by tests/test_host_rules.py.
#include <cstdio>
#include <cstring>
#include <vector>

#include "hip/ccd_rules.hpp"
#include "hip/pcg_rules.hpp"
#include "hip/pcg_words.hpp"

using namespace silk::amd;

#define CHECK(c)                                              \
  do {                                                        \
    if (!(c)) {                                               \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);     \
      return 1;                                               \
    }                                                         \
  } while (0)

// Every place the kernel reads lies in the table, whatever slices have no
// entries: the table is as long as its slices, and one entry long when none
// has any.
static int sell() {
  constexpr int kSlice = 64, kNbr = 32;
  for (const std::vector<int>& widths :
       {std::vector<int>{0}, {0, 0}, {8, 0}, {0, 8}, {16, 0, 8, 0, 0}, {40, 0}, {32}}) {
    std::vector<int> off;
    int size = 0;
    for (int w : widths) {
      off.push_back(size);
      size += w * kSlice;
    }
    const int table = size > 0 ? size : 1;
    for (size_t s = 0; s < widths.size(); ++s)
      for (int lane = 0; lane < kSlice; ++lane)
        for (int e = 0; e < kNbr; ++e) {
          const int at = sell_place(off[s], widths[s], e, kSlice, lane);
          CHECK(at >= 0 && at < table);
          if (e < widths[s]) CHECK(at == off[s] + e * kSlice + lane);
        }
  }
  return 0;
}

template <class T>
struct HostBuf {
  std::vector<T> v;
  void zero(int) { v.assign(v.size(), T(0)); }
};

// Every buffer is listed, and none keeps a word (a tag of an epoch that will be
// handed out again, a counter, the flag) when they are cleared.
static int clear() {
  PcgWords<HostBuf> w;
  size_t n = 0;
  w.each([&](auto& b) {
    b.v.assign(10 + n++, 1u);
  });
  CHECK(sizeof(w) == n * sizeof(HostBuf<int>));
  w.clear(0);
  size_t words = 0;
  int left = 0;
  w.each([&](auto& b) {
    for (auto x : b.v) left += x != 0;
    words += b.v.size();
  });
  CHECK(left == 0 && words == 10 * n + n * (n - 1) / 2);
  return 0;
}

// The tags of one level-1 sum through 300,000 solves that end at their first
// exchange, with and without the true-residual test's two exchanges, each
// followed by a solve of several steps: what lies in a buffer never carries
// the 16 bits of the epoch that is waited for, and no epoch is used twice.
static int epochs() {
  for (int test : {0, 2}) {
    unsigned tag[2] = {0, 0}, counter = 0, highest = 0;
    for (int solve = 0; solve < 300000; ++solve) {
      unsigned ep = counter;
      const int exchanges = solve % 32768 == 32767 || solve == 0 ? 4 : 1;
      for (int k = 0; k < exchanges; ++k) {
        ++ep;
        CHECK(ep > highest);
        CHECK((tag[ep & 1] & 0xffffu) != (ep & 0xffffu));
        tag[ep & 1] = ep;
        highest = ep + 1;  // M0 r of the next exchange goes out early
        if (k + 1 < exchanges) highest = ep;
      }
      ep += static_cast<unsigned>(test);
      counter = one_last_epoch(counter, ep);
    }
  }
  return 0;
}

// Passes that count for one, for two, and for both in turn: the minimum is
// re-read within 33 counts of the last time, and not before 32.
static int refresh() {
  for (int pattern = 0; pattern < 4; ++pattern) {
    CutRefresh r;
    int last = 0;
    for (int pass = 0, iter = 1; iter < 4000; ++pass) {
      const bool due = r.due(iter);
      if (due) CHECK(iter - last >= 32);
      if (due) last = iter;
      CHECK(iter - last < 34);
      iter += pattern == 0 ? 1 : pattern == 1 ? 2 : pattern == 2 ? 1 + pass % 2 : 1 + pass % 3 / 2;
    }
  }
  return 0;
}

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  if (std::strcmp(argv[1], "sell") == 0) return sell();
  if (std::strcmp(argv[1], "clear") == 0) return clear();
  if (std::strcmp(argv[1], "epochs") == 0) return epochs();
  if (std::strcmp(argv[1], "refresh") == 0) return refresh();
  return 2;
}
