// The passes that a run of ticks takes on a world's bit planes, and what holds about
// the planes between calls.  Host code without device calls: the launches are the
// caller's (Ops), so that the bookkeeping can be checked without a device.
#pragma once

#include <cstdint>

namespace fs3d {

// What a pass over the active items must know of the flags before it: those of a pass
// like it, none (the grid has just been packed: every flag is set), or those of packing
// and ticking in one pass (plane.h).  kNoFlags: there is nothing to read.
enum { kNotFirst = 0, kAfterPack, kAfterPackTick, kNoFlags };
constexpr int kFlagBufs = 3;  // the last pass's, the one before's, and the next one's
inline int next_flags(int f) { return f + 1 < kFlagBufs ? f + 1 : 0; }

// A world's planes between calls.
struct PlaneState {
  bool valid = false;  // planes[cur] holds the current state
  bool tiled = false;  // the layout of the buffers
  int cur = 0;
  int flags = 0;           // the last pass's flag buffer and the next one's list counter,
  int first = kAfterPack;  // and what the next pass must know of those flags: a pass that has
                           // only packed and ticked leaves others than one over the items
  int older = kNoFlags;    // the same for the flags of the pass before it.  A block rests when
                           // neither parity's last tick changed it or a cell of it, so
                           // behind a pass of one tick the one before counts too.
  int shorts = 0;          // runs under kPlaneMinTicks ticks since the last longer one
  bool ready(bool want_tiled) const { return valid && tiled == want_tiled; }
  // The next tick has the parity of the last one: the other parity's last tick is not
  // among the flags.
  void parity_repeats() {
    first = kAfterPack;
    older = kNoFlags;
  }
};

// Whether a run takes the planes (a grid that can be in planes; items: passes over the
// active items only) or stays on bytes.
//
// Packing and unpacking everything cost about a byte tick each (512^3: 24 + 42 us), so
// runs under three ticks do not pay for them, nor for the unpacking alone: one tick of a
// grid in planes takes 193 us at 800^3, on bytes 57 with columns falling and 24 at rest
// (512^3: 37 against 27 and 11; 64^3: 16 against 7).
//
// With items, only what moved is unpacked, but a single tick still takes more than on
// bytes (1024^3, columns: 103 against 72 us; at rest 50 against 27), while going to bytes
// and back takes two ticks of everything and a packing, 0.8 ms.  So such a run stays in
// planes until 24 of them in a row have wasted that much.  (A hash per tick is cheaper on
// planes: 320 against 407 us.)
constexpr int kPlaneMinTicks = 3, kPlaneShortRuns = 24;

// The hash of planes takes longer than the one a byte tick takes as it writes, which tells
// where the byte ticks run in place and in the last-level cache (512^3 boxes: 117 against
// 72 us).  us per tick with a hash after every one, bytes / planes, boxes and rain:
//   256^3 26, 13 / 25, 15     320^3 37, 19 / 40, 23     512^3 101, 52 / 127, 55
//   560^3 216, 110 / 160, 71  (200^3 20, 13 / 18, 12)
// and after every second one, where a skipping world's byte ticks are cheap: 320^3 rain
// 12 / 15, 512^3 30 / 32.  A word of a row under 24 cells is mostly padding, which the hash
// walks too: 16 x 1024 x 1024, hash after every tick / sixth tick / none, 26, 12, 8 on
// bytes, 67, 17, 8 on planes.
constexpr uint64_t kHashedBytesMin = 3ull << 22, kHashedBytesMax = 1ull << 27, kNarrowMin = 1ull << 21;
constexpr int kNarrowRow = 24;

struct PlaneRun {
  uint64_t n;  // voxels
  int nx;
  bool skip, items;
  int nticks, hash_every;
};
inline bool planes_suit(const PlaneState &st, const PlaneRun &r) {
  const int64_t hashes = r.hash_every > 0 ? r.nticks / r.hash_every : 0;
  if (r.nticks < kPlaneMinTicks) return r.items && st.ready(true) && (hashes || st.shorts < kPlaneShortRuns);
  if (r.nx < kNarrowRow && r.n > kNarrowMin && 6 * hashes >= r.nticks) return false;
  const bool often = r.skip ? 2 * hashes >= r.nticks : 2 * hashes > r.nticks;
  return !(often && r.n > kHashedBytesMin && r.n <= kHashedBytesMax);
}

// A pass: one tick, or the ticks t (odd) and t + 1.
struct PlanePass {
  int k;       // ticks of the run before it
  bool pair;
  int src;     // reads planes[src], writes planes[src ^ 1]
  int flags;   // items: reads flag buffer `flags` (and the one before it), writes the next one,
               // appends to counter `flags` and clears the next one
  int first, older;  // items: kNotFirst, ...
  int hash;    // everything: the hash (1, 2, ...) of planes[src] taken in the same launch, or 0
};

// nticks ticks from tick t0 with a hash every hash_every (0: none); items: passes over
// the active items only.  *st becomes the state after them.  Ops, each returning 0 or
// an error:
//   packed(items)            the grid is about to be packed; items: clears the counters
//   pack(src)                bytes to planes[src]
//   pack_tick(src, flags)    the same and tick t0 (even); flags: -1 or the flag buffer to write
//   all_flags(flags)         every flag set
//   zero_hashes(n)
//   hash(src, i)             hash i of planes[src]
//   pass(p), item_pass(p)
//   unpack(src, flags)       planes[src] to bytes; flags: -1 or the last pass's flag buffer
template <class Ops>
int plane_passes(PlaneState *st, bool items, uint64_t t0, int nticks, int hash_every, Ops &&ops) {
  int src = st->valid ? st->cur : 0, f = st->flags;
  // an even first tick is done while packing
  const bool packs = !st->valid, ticks_too = packs && !(t0 & 1u);
  st->valid = false;  // should a launch fail, the bytes are the state
  int first = ticks_too ? kAfterPackTick : packs ? kAfterPack : st->first;
  int older = packs ? kNoFlags : st->older;
  if (packs) {
    if (int rc = ops.packed(items)) return rc;
    if (int rc = ticks_too ? ops.pack_tick(src, items ? f : -1) : ops.pack(src)) return rc;
  }
  if (items && first == kAfterPack)
    if (int rc = ops.all_flags(f)) return rc;
  auto hashed_after = [&](int k) { return hash_every > 0 && (k + 1) % hash_every == 0; };
  if (hash_every > 0 && nticks >= hash_every)
    if (int rc = ops.zero_hashes(nticks / hash_every)) return rc;
  int due = ticks_too && hashed_after(0) ? 1 : 0;  // the hash that planes[src] has yet to give
  for (int k = ticks_too ? 1 : 0; k < nticks;) {
    const bool pair = ((t0 + (uint64_t)k) & 1u) && k + 1 < nticks && !hashed_after(k);
    // a single tick hashes the state that it reads
    const bool with = due && !items && !pair;
    if (due && !with)
      if (int rc = ops.hash(src, due)) return rc;
    const PlanePass p{k, pair, src, f, first, older, with ? due : 0};
    if (int rc = items ? ops.item_pass(p) : ops.pass(p)) return rc;
    src ^= 1;
    if (items) f = next_flags(f);  // (a pass over everything clears no counter)
    older = pair ? (int)kNoFlags : first == kAfterPackTick ? (int)kAfterPackTick : (int)kNotFirst;
    first = kNotFirst;
    k += pair ? 2 : 1;
    due = hashed_after(k - 1) ? k / hash_every : 0;
  }
  if (due)
    if (int rc = ops.hash(src, due)) return rc;
  if (int rc = ops.unpack(src, items ? f : -1)) return rc;
  st->cur = src;
  st->valid = true;
  st->shorts = nticks >= kPlaneMinTicks ? 0 : st->shorts + 1;
  st->flags = f;
  st->first = items ? first : (int)kAfterPack;
  st->older = items ? older : (int)kNoFlags;
  return 0;
}

}  // namespace fs3d
