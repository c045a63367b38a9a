// Which items a pass over the active items visits (plane.hip has the rule and the
// flags' meaning).  Host and device code.
#pragma once

#include <cstddef>
#include <cstdint>

#include "plane_core.h"
#include "plane_sched.h"

namespace fs3d {
namespace plane {

typedef uint64_t u64;

// Flags are u64 masks over the words of a strip (bit = word), kFlags per cell of the strip
// grid, each flag of all cells in a row: any change; a change of a block at the item's
// first or last word bit, row, layer; any change in the last pass alone.
enum { kAny = 0, kXFirst, kXLast, kYFirst, kYLast, kZFirst, kZLast, kNow, kFlags };

// The words of cell (st, zr) with work, by the flags of the pass before: an item that
// changed, and its neighbours across the faces at which it did.
FS3D_HD u64 plan_words(const u64 *in, int strips, int zcells, int st, int zr, int first) {
  const size_t ncell = (size_t)strips * (size_t)zcells;
  u64 act = 0;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
  for (int dz = -1; dz <= 1; dz++)
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
    for (int dy = -1; dy <= 1; dy++) {
      const int y = st + dy, z = zr + dz;
      if (y < 0 || y >= strips || z < 0 || z >= zcells) continue;
      const u64 *f = in + ((size_t)z * strips + y);
      u64 m = f[kAny];
      if (m == 0) continue;
      if (first == kAfterPackTick) {  // what can move in an item may touch all its sides
        act |= m | (m >> 1) | (m << 1);
        continue;
      }
      if (dy) m &= f[(size_t)(dy > 0 ? kYFirst : kYLast) * ncell];
      if (dz) m &= f[(size_t)(dz > 0 ? kZFirst : kZLast) * ncell];
      act |= m | ((m & f[(size_t)kXFirst * ncell]) >> 1) | ((m & f[(size_t)kXLast * ncell]) << 1);
    }
  return act;
}

// The flags of cell c before the pass adds to them, and the items changed since the bytes
// were written, to which the pass before adds its changes.
FS3D_HD void plan_flags(const u64 *in, u64 *out, u64 *since, size_t c, size_t ncell, int first) {
  const u64 now = first == kAfterPack ? 0 : in[(size_t)kNow * ncell + c];
  if (first != kNotFirst)
    since[c] = now;
  else if (now)
    since[c] |= now;
  for (int i = 0; i < kFlags; i++) out[(size_t)i * ncell + c] = 0;
}

}  // namespace plane
}  // namespace fs3d
