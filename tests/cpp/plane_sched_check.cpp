// The bookkeeping of the passes over a world's bit planes, without a device: list
// counters through changes between passes over the active items and over everything.
#include <cstdio>
#include <random>

#include "../../fallingsand3d_amd/csrc/plane_sched.h"

using namespace fs3d;

#define CHECK(c)                                        \
  do {                                                  \
    if (!(c)) {                                         \
      std::printf("FAILED line %d: %s\n", __LINE__, #c); \
      return 1;                                         \
    }                                                   \
  } while (0)

// Counts as the kernels do: the plan appends to the pass's counter, the pass reads it
// and clears the other one.
struct Counters {
  unsigned n[2] = {0, 0};
  unsigned items = 100;
  int packed(bool items) {
    if (items) n[0] = n[1] = 0;
    return 0;
  }
  int pack(int) { return 0; }
  int pack_tick(int, int) { return 0; }
  int all_flags(int) { return 0; }
  int zero_hashes(int) { return 0; }
  int hash(int, int) { return 0; }
  int pass(const PlanePass &) { return 0; }
  int item_pass(const PlanePass &p) {
    CHECK(n[p.flags] == 0);
    n[p.flags] += items;
    n[p.flags ^ 1] = 0;
    return 0;
  }
  int unpack(int, int) { return 0; }
};

// A world's calls: the layout of the planes is dropped when the schedule changes.
static int counters() {
  for (unsigned t0 = 0; t0 < 2; t0++)
    for (int dense = 1; dense < 6; dense++)
      for (int n = 1; n < 5; n++) {
        Counters ops;
        PlaneState st;
        uint64_t t = t0;
        auto run = [&](bool items, int n) {
          const int rc = plane_passes(&st, items, t, n, 0, ops);
          t += (uint64_t)n;
          return rc;
        };
        for (int k = 0; k < 3; k++) {
          CHECK(run(true, 3 + k) == 0);
          st.valid = false;
          CHECK(run(false, dense) == 0);
          st.valid = false;
          CHECK(run(true, n) == 0);
        }
      }
  return 0;
}

int main() {
  if (counters()) return 1;
  std::printf("plane schedule checks passed\n");
  return 0;
}
