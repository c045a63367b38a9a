// Internal declarations of the bit-plane kernels (plane.hip).
#pragma once

#include <algorithm>

#include "fs3d_internal.h"

namespace fs3d {

typedef u32 plane_u32x4 __attribute__((ext_vector_type(4)));

// Rows of words with a row of zeros before every layer and layers of them at the ends
// (plane.hip); or tiled, for the ticks of active items: eight rows' words of a column
// side by side, 128 bytes of memory for 64 x 8 cells instead of 512 x 1.
struct PlaneShape {
  int nx = 0, ny = 0, nz = 0;
  int lr = 0;  // 64-cell words per row
  bool tiled = false;
};
inline PlaneShape plane_shape(int nx, int ny, int nz, bool tiled = false) {
  return PlaneShape{nx, ny, nz, (nx + 63) / 64, tiled};
}
// Tiles along y: one before row 0, so that four strips of an even tick's row quads are
// a tile, and rows 0 .. ny + 1.
inline int plane_tiles(const PlaneShape &p) { return (p.ny + 9) / 8 + 1; }
// 16-byte words of a plane grid with the zero rows around it.
inline size_t plane_words(const PlaneShape &p) {
  if (p.tiled) return (size_t)p.lr * 8 * (size_t)plane_tiles(p) * (size_t)(p.nz + 2);
  return (size_t)p.lr * ((size_t)(p.ny + 1) * (size_t)(p.nz + 2) + 1);
}

// Workgroups of a single tick (one at least for every two layers, however thin they are).
// A launch takes fewer than 2^32 threads; half of that is the tick's, the rest room for
// the hash in the same launch.
inline u64 plane_tick_rows(const PlaneShape &p) {  // workgroups along y
  const u64 per = 4 * (64 / (u64)p.lr), nyq = ((u64)p.ny + 2) >> 1;
  return (nyq + per - 1) / per;
}
inline u64 plane_tick_blocks(const PlaneShape &p) { return plane_tick_rows(p) * (((u64)p.nz + 2) >> 1); }
constexpr u64 kMaxTickBlocks = 1ull << 23;

struct PlaneArgs {
  const plane_u32x4 *src;
  plane_u32x4 *dst;
  u32 bytes;  // of a plane grid (< 4 GiB)
  int ny, nz, lr;
  int upw;       // units (row quads or strips of them) per wave
  u32 lr_magic;  // lane / lr = (lane * lr_magic) >> 16
  u64 t;
  const u64 *tick_dev;  // when set, tick = *tick_dev + k_off (graph replays)
  u32 k_off;
  int zlen, ytiles;  // pairs: z row-quads per wave, waves along y
};

// State hash of a grid; g holds the bytes of reserved cells.  With plane_hash_direct
// it is added to *out, otherwise to the partial sums, which launch_hash_finalize adds
// up.
struct PlaneHash {
  const u8 *g;
  const u32 *reserved;
  u64 *parts, *out;
};
bool plane_hash_direct(const PlaneShape &ps);
hipError_t launch_plane_hash(const PlaneShape &ps, const void *planes, const PlaneHash &hash, hipStream_t s);
// One tick, any parity, and the hash of src when asked for.
hipError_t launch_plane_tick(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             const PlaneHash *hash, hipStream_t s);
// Ticks t and t + 1, t odd.
hipError_t launch_plane_pair(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             hipStream_t s);
// Zeroes the rows around the grid (no kernel here writes them).
hipError_t launch_plane_pad(const PlaneShape &ps, void *planes, hipStream_t s);
// Bytes (values >= 4 as STATIC, *reserved set) to planes and back (with *reserved,
// bytes >= 4 already in g stay).
hipError_t launch_plane_pack(const PlaneShape &ps, const u8 *g, void *planes, u32 *reserved, hipStream_t s);
// Packing and the even tick t on it: planes hold the state after the tick, flags
// (of items; or nullptr) what the next pass needs with kAfterPackTick; other: the
// buffer that it will write.
hipError_t launch_plane_pack_even(const PlaneShape &ps, const u8 *g, void *planes, u32 *reserved, u64 t,
                                  const u64 *tick_dev, u32 k_off, u64 *flags, void *other, hipStream_t s);
hipError_t launch_plane_unpack(const PlaneShape &ps, const void *planes, u8 *g, const u32 *reserved, hipStream_t s);

// The word that holds a cell.
size_t plane_word(const PlaneShape &ps, int x, int y, int z);

// ---- ticks of the active items only (plane.hip has the rule) ----
constexpr int kItemQuads = 1;   // even-parity row quads of an item along y
constexpr int kItemLayers = 8;  // and along z
struct PlaneCells {
  int strips = 0, zcells = 0;  // the strip grid: items of one word per cell and word
  int virt = 0;                // 1: a virtual word behind each row
  size_t flag_words = 0, since_words = 0, list_words = 0;  // u64, u64, u32
};
PlaneCells plane_cells(const PlaneShape &ps);
// Where the change flags of a cell's item begin (*n of them, *stride apart, bit = word).
size_t plane_cell_flags(const PlaneShape &ps, int y, int z, int *n, size_t *stride);
int plane_list_blocks_per_cu();
// A pass over the active items: ticks t and t + 1 (pair, t odd) or tick t (of
// either parity; *tick_dev + k_off has t's).  flags_in: the pass before, older: the one
// before that, where the pass before ran one tick (else nullptr); flags_out: this one's;
// since: items changed since the bytes were written; first and older_first: kAfterPack
// for the flags after packing (every one set), kAfterPackTick for those of
// launch_plane_pack_even.  *count is 0 before; the pass clears *next_count.
hipError_t launch_plane_list(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             bool pair, int first, const u64 *flags_in, int older_first, const u64 *older,
                             u64 *flags_out, u64 *since, u32 *list, u32 *count, u32 *next_count, u32 nwaves,
                             hipStream_t s);
// Writes the bytes of the items in since or flags (the last pass's) and clears since;
// dirty (or nullptr): a bit per 8^3 brick, set for those that hold a written item.
hipError_t launch_plane_unpack_cells(const PlaneShape &ps, const void *planes, u8 *g, const u64 *flags, u64 *since,
                                     const u32 *reserved, u64 *dirty, hipStream_t s);

}  // namespace fs3d
