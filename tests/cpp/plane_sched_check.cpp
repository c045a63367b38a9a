// The bookkeeping of the passes over a world's bit planes, without a device: list
// counters through changes between passes over the active items and over everything,
// and a model of such a world, cell by cell, whose passes write nothing but the items that
// the plan lists.  Reads the rule table (4 x 65536 u16, lut[v * 65536 + s]) from argv[1].
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "../../fallingsand3d_amd/csrc/plane_plan.h"

using namespace fs3d;
using plane::u64;
typedef unsigned char u8;

#define CHECK(c)                                         \
  do {                                                   \
    if (!(c)) {                                          \
      std::printf("FAILED line %d: %s\n", __LINE__, #c); \
      return 1;                                          \
    }                                                    \
  } while (0)

// ---- list counters ----
// The plan appends to the pass's counter, the pass reads it and clears the next one.
struct Counters {
  unsigned n[kFlagBufs] = {};
  unsigned items = 100;
  int packed(bool with_items) {
    if (with_items)
      for (unsigned &c : n) c = 0;
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
    n[next_flags(p.flags)] = 0;
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
        u64 t = t0;
        auto run = [&](bool items, int ticks) {
          const int rc = plane_passes(&st, items, t, ticks, 0, ops);
          t += (u64)ticks;
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

// ---- a world ----
static std::vector<uint16_t> lut;

struct Model {
  // items of one 64-cell word, 2 rows and 16 layers
  static constexpr int IX = 64, IY = 2, IZ = 16;
  int nx, ny, nz, lr, strips, zcells;
  size_t ncell;
  std::vector<u8> bytes, buf[2];
  std::vector<u64> flags[kFlagBufs], since;
  PlaneState st;
  bool items = true;
  u64 t = 0;
  bool any_path = false;  // in planes whenever the grid is there, as a long run would
  long listed = 0;        // words of the last pass over the items

  Model(int x, int y, int z) : nx(x), ny(y), nz(z) {
    lr = (nx + 63) / 64;
    strips = (ny + 1) / 2;
    zcells = ((nz + 1) / 2 + 7) / 8;
    ncell = (size_t)strips * zcells;
    bytes.assign((size_t)nx * ny * nz, 0);
    for (auto &b : buf) b.assign(bytes.size(), 9);
    for (auto &f : flags) f.assign(ncell * plane::kFlags, 0x5555);
    since.assign(ncell, 0);
  }
  size_t at(int x, int y, int z) const { return ((size_t)z * ny + y) * nx + x; }
  size_t cell(int y, int z) const { return (size_t)(z / IZ) * strips + y / IY; }

  // One tick of every block; f (when not null) receives the flags of the items that a
  // changed block touches, as far as the pass has listed them.
  void tick(const std::vector<u8> &in, std::vector<u8> &out, u64 tt, std::vector<u64> *f,
            const std::vector<u64> *act) const {
    const int p = (int)(tt & 1);
    out = in;
    for (int z0 = -p; z0 < nz; z0 += 2)
      for (int y0 = -p; y0 < ny; y0 += 2)
        for (int x0 = -p; x0 < nx; x0 += 2) {
          unsigned s = 0;
          for (int c = 0; c < 8; c++) {
            const int x = x0 + (c & 1), y = y0 + ((c >> 1) & 1), z = z0 + (c >> 2);
            const bool in_grid = x >= 0 && y >= 0 && z >= 0 && x < nx && y < ny && z < nz;
            s |= (in_grid ? in[at(x, y, z)] : 1u) << (2 * c);
          }
          const unsigned v = plane::mix32((unsigned)(x0 * 7919 + y0 * 104729 + z0 * 1299709) + (unsigned)tt) & 3u;
          const unsigned r = lut[v * 65536 + s];
          if (r == s) continue;
          for (int c = 0; c < 8; c++) {
            const int x = x0 + (c & 1), y = y0 + ((c >> 1) & 1), z = z0 + (c >> 2);
            if (x < 0 || y < 0 || z < 0 || x >= nx || y >= ny || z >= nz) continue;
            out[at(x, y, z)] = (r >> (2 * c)) & 3u;
            if (!f) continue;
            const size_t i = cell(y, z);
            const u64 bit = 1ull << (x / IX);
            if (!((*act)[i] & bit)) continue;
            auto set = [&](int kind) { (*f)[(size_t)kind * ncell + i] |= bit; };
            set(plane::kAny);
            set(plane::kNow);
            // the block is at a face when it holds cells of the item's first or last
            // block along the axis
            const int wx = x / IX * IX, wy = y / IY * IY, wz = z / IZ * IZ;
            if (x0 <= wx) set(plane::kXFirst);
            if (x0 + 1 >= wx + IX - 1) set(plane::kXLast);
            if (y0 <= wy) set(plane::kYFirst);
            if (y0 + 1 >= wy + IY - 1) set(plane::kYLast);
            if (z0 <= wz) set(plane::kZFirst);
            if (z0 + 1 >= wz + IZ - 1) set(plane::kZLast);
          }
        }
  }

  template <class Fn>
  void each(const std::vector<u64> &act, Fn &&fn) const {
    for (int z = 0; z < nz; z++)
      for (int y = 0; y < ny; y++)
        for (int x = 0; x < nx; x++)
          if ((act[cell(y, z)] >> (x / IX)) & 1) fn(at(x, y, z));
  }

  int packed(bool) { return 0; }
  int pack(int src) {
    buf[src] = bytes;
    buf[src ^ 1].assign(bytes.size(), 9);
    return 0;
  }
  int pack_tick(int src, int f) {
    buf[src ^ 1].assign(bytes.size(), 9);
    tick(bytes, buf[src], t, nullptr, nullptr);
    if (f < 0) return 0;
    flags[f].assign(flags[f].size(), 0);
    std::vector<u64> still(ncell, (1ull << lr) - 1);
    for (int z = 0; z < nz; z++)
      for (int y = 0; y < ny; y++)
        for (int x = 0; x < nx; x++) {
          const u64 bit = 1ull << (x / IX);
          const size_t i = cell(y, z);
          if (buf[src][at(x, y, z)] >= 2) flags[f][plane::kAny * ncell + i] |= bit, still[i] &= ~bit;
          if (buf[src][at(x, y, z)] != bytes[at(x, y, z)]) flags[f][plane::kNow * ncell + i] |= bit;
        }
    each(still, [&](size_t i) { buf[src ^ 1][i] = buf[src][i]; });
    return 0;
  }
  int all_flags(int f) {
    flags[f].assign(flags[f].size(), ~0ull);
    return 0;
  }
  int zero_hashes(int) { return 0; }
  int hash(int, int) { return 0; }
  int pass(const PlanePass &p) {
    std::vector<u8> s;
    tick(buf[p.src], s, t + (u64)p.k, nullptr, nullptr);
    if (p.pair)
      tick(s, buf[p.src ^ 1], t + (u64)p.k + 1, nullptr, nullptr);
    else
      buf[p.src ^ 1] = s;
    return 0;
  }
  int item_pass(const PlanePass &p) {
    const std::vector<u64> &in = flags[p.flags], &older = flags[next_flags(next_flags(p.flags))];
    std::vector<u64> act(ncell, 0), *out = &flags[next_flags(p.flags)];
    const u64 words = (1ull << lr) - 1;
    listed = 0;
    for (int z = 0; z < zcells; z++)
      for (int y = 0; y < strips; y++) {
        const size_t c = (size_t)z * strips + y;
        act[c] = plane::plan_words(in.data(), strips, zcells, y, z, p.first);
        if (p.older != kNoFlags) act[c] |= plane::plan_words(older.data(), strips, zcells, y, z, p.older);
        act[c] &= words;
        listed += __builtin_popcountll(act[c]);
      }
    for (size_t c = 0; c < ncell; c++)
      plane::plan_flags(in.data(), out->data(), since.data(), c, ncell, p.first);
    std::vector<u8> s1, s2;
    tick(buf[p.src], s1, t + (u64)p.k, out, &act);
    if (p.pair)
      tick(s1, s2, t + (u64)p.k + 1, out, &act);
    else
      s2 = s1;
    each(act, [&](size_t i) { buf[p.src ^ 1][i] = s2[i]; });
    CHECK(buf[p.src ^ 1] == s2);  // what is not listed is what the buffer held
    return 0;
  }
  int unpack(int src, int f) {
    if (f < 0) {
      bytes = buf[src];
      return 0;
    }
    std::vector<u64> act(ncell);
    for (size_t c = 0; c < ncell; c++) act[c] = since[c] | flags[f][plane::kNow * ncell + c], since[c] = 0;
    each(act, [&](size_t i) { bytes[i] = buf[src][i]; });
    CHECK(bytes == buf[src]);
    return 0;
  }

  // a world's calls
  int run(int n, int every) {
    const std::vector<u8> before = bytes;
    if (any_path ? st.ready(items) || n >= kPlaneMinTicks : planes_suit(st, {bytes.size(), nx, items, items, n, every})) {
      if (st.tiled != items) {
        st.tiled = items;
        st.valid = false;
      }
      if (plane_passes(&st, items, t, n, every, *this)) return 1;
    } else {
      st.valid = false;
      for (int k = 0; k < n; k++) {
        std::vector<u8> s;
        tick(bytes, s, t + (u64)k, nullptr, nullptr);
        bytes = s;
      }
    }
    std::vector<u8> want = before, s;
    for (int k = 0; k < n; k++, want = s) tick(want, s, t + (u64)k, nullptr, nullptr);
    t += (u64)n;
    CHECK(bytes == want);
    return 0;
  }
  void set_tick(u64 tick) {
    if ((tick ^ t) & 1) st.parity_repeats();
    t = tick;
  }
  void poke(int x, int y, int z, u8 v) {
    bytes[at(x, y, z)] = v;
    if (!st.valid) return;
    buf[st.cur][at(x, y, z)] = v;
    if (st.first == kAfterPack) return;
    for (int i = 0; i < plane::kFlags; i++) flags[st.flags][(size_t)i * ncell + cell(y, z)] |= 1ull << (x / IX);
  }
  void fill(std::mt19937 &rng) {
    // sand and fluid in a few clumps over a floor: most items rest
    for (size_t i = 0; i < bytes.size(); i++) bytes[i] = i < (size_t)nx * ny ? 1 : 0;
    for (int k = 0; k < 6; k++) {
      const int cx = (int)(rng() % nx), cy = (int)(rng() % ny), cz = (int)(rng() % nz);
      for (int z = cz; z < std::min(nz, cz + 9); z++)
        for (int y = cy; y < std::min(ny, cy + 4); y++)
          for (int x = cx; x < std::min(nx, cx + 7); x++)
            if (z > 0 && rng() % 3) bytes[at(x, y, z)] = (u8)(1 + rng() % 3);
    }
    st.valid = false;
  }
};

// What an interactive program does: runs, single ticks, pokes, changes of schedule.
static int worlds() {
  for (unsigned seed = 1; seed <= 40; seed++) {
    std::mt19937 rng(seed);
    Model w(seed & 1 ? 150 : 192, 9, 37 + (int)(seed % 3));
    w.any_path = seed % 4 < 2;
    w.t = seed % 2;
    w.fill(rng);
    for (int k = 0; k < 25; k++) {
      switch (rng() % 10) {
        case 0: w.items = !w.items; break;
        case 1:
          for (int i = 0; i < 5; i++)
            w.poke((int)(rng() % w.nx), (int)(rng() % w.ny), (int)(rng() % w.nz), (u8)(rng() % 4));
          break;
        case 2:
          if (rng() % 3 == 0) w.fill(rng);
          break;
        case 3: w.set_tick(w.t + rng() % 3); break;
        default: CHECK(w.run(1 + (int)(rng() % 6), (int)(rng() % 3)) == 0);
      }
    }
  }
  return 0;
}

// A single tick right after the schedule has changed, from either parity.
static int switches() {
  for (unsigned t0 = 0; t0 < 2; t0++)
    for (int n = 1; n < 4; n++) {
      std::mt19937 rng(t0 + 7);
      Model w(192, 9, 38);
      w.t = t0;
      w.any_path = true;
      w.fill(rng);
      w.items = false;
      CHECK(w.run(10, 0) == 0);
      w.items = true;
      for (int k = 0; k < 12; k++) CHECK(w.run(n, 0) == 0);
      w.items = false;
      CHECK(w.run(3, 0) == 0);
      w.items = true;
      for (int k = 0; k < 12; k++) CHECK(w.run(n, 0) == 0);
    }
  return 0;
}

// What has come to rest is left alone, however the ticks are taken.
static int rest() {
  for (int every = 0; every < 2; every++)
    for (int n : {1, 2, 5}) {
      std::mt19937 rng(5);
      Model w(192, 9, 38);
      w.any_path = true;
      w.fill(rng);
      for (u8 &c : w.bytes) c = c == 3 ? 0 : c;  // sand comes to rest
      for (int k = 0; k < 150; k += n) CHECK(w.run(k < 3 ? 3 : n, every) == 0);
      CHECK(w.listed == 0);
      w.poke(100, 4, 30, 2);
      for (int k = 0; k < 4; k++) CHECK(w.run(n, every) == 0);
      CHECK(w.listed > 0 && w.listed < 30);
    }
  return 0;
}

// Which runs take the planes.
static int paths() {
  auto suits = [](const PlaneState &st, u64 n, int nx, bool skip, int ticks, int every) {
    return planes_suit(st, {n, nx, skip, skip && n > 1ull << 28, ticks, every});
  };
  const u64 big = 1ull << 29, mid = 1ull << 26;
  PlaneState dense, items;
  for (bool skip : {false, true})
    for (int n : {1, 2}) {
      CHECK(!suits(dense, mid, 500, skip, n, 0) && !suits(items, big, 500, true, n, 0));
      dense.valid = true;  // in planes, which are no better for them
      CHECK(!suits(dense, mid, 500, skip, n, 0) && !suits(dense, 4000, 500, skip, n, 1));
      dense.valid = false;
    }
  CHECK(suits(dense, mid, 500, true, 3, 0) && suits(items, big, 500, true, 3, 0));
  Counters ops;
  items.tiled = true;
  CHECK(plane_passes(&items, true, 0, 4, 0, ops) == 0);
  int k = 0;  // single ticks on planes before they go to bytes
  for (; k < 1000 && suits(items, big, 500, true, 1, 0); k++) CHECK(plane_passes(&items, true, (u64)k, 1, 0, ops) == 0);
  CHECK(k == kPlaneShortRuns && suits(items, big, 500, true, 1, 1) && suits(items, big, 500, true, 3, 0));
  CHECK(plane_passes(&items, true, (u64)k, 3, 0, ops) == 0 && suits(items, big, 500, true, 1, 0));
  // hashed often: on bytes where those run in the last-level cache
  for (bool skip : {false, true}) {
    CHECK(!suits(dense, mid, 500, skip, 30, 1) && !suits(dense, 1ull << 27, 500, skip, 30, 1));
    CHECK(!suits(dense, (3ull << 22) + 1, 500, skip, 30, 1) && suits(dense, 3ull << 22, 500, skip, 30, 1));
    CHECK(suits(dense, (1ull << 27) + 1, 500, skip, 30, 1));
    CHECK(suits(dense, mid, 500, skip, 30, 2) == !skip && suits(dense, mid, 500, skip, 30, 3));
    CHECK(suits(dense, mid, 500, skip, 30, 30));
    // rows that are mostly padding
    CHECK(!suits(dense, 1ull << 22, 16, skip, 30, 6) && !suits(dense, big, 23, skip, 30, 1));
    CHECK(suits(dense, 1ull << 21, 16, skip, 30, 6) && suits(dense, 1ull << 22, 16, skip, 30, 7));
    CHECK(suits(dense, 1ull << 22, 24, skip, 30, 1) && suits(dense, 1ull << 22, 16, skip, 30, 0));
  }
  return 0;
}

int main(int argc, char **argv) {
  if (argc < 2) return 2;
  lut.resize(4 * 65536);
  FILE *f = std::fopen(argv[1], "rb");
  if (!f || std::fread(lut.data(), 2, lut.size(), f) != lut.size()) return 2;
  std::fclose(f);
  if (counters() || paths() || switches() || rest() || worlds()) return 1;
  std::printf("plane schedule checks passed\n");
  return 0;
}
