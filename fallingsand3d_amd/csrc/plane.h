// Internal declarations of the bit-plane kernels (plane.hip).
#pragma once

#include <algorithm>

#include "fs3d_internal.h"

namespace fs3d {

typedef u32 plane_u32x4 __attribute__((ext_vector_type(4)));

struct PlaneShape {
  int nx = 0, ny = 0, nz = 0;
  int lr = 0;  // 64-cell words per row
};
inline PlaneShape plane_shape(int nx, int ny, int nz) { return PlaneShape{nx, ny, nz, (nx + 63) / 64}; }
// 16-byte words of a plane grid.
inline size_t plane_words(const PlaneShape &p) { return (size_t)p.lr * (size_t)p.ny * (size_t)p.nz; }

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

// One tick, any parity.
hipError_t launch_plane_tick(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             hipStream_t s);
// Ticks t and t + 1, t odd: k even-parity row quads along y and zlen along z per lane.
hipError_t launch_plane_pair(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             int k, int zlen, hipStream_t s);
// Bytes (values >= 4 as STATIC, *reserved set) to planes and back (with *reserved,
// bytes >= 4 already in g stay).
hipError_t launch_plane_pack(const PlaneShape &ps, const u8 *g, void *planes, u32 *reserved, hipStream_t s);
hipError_t launch_plane_unpack(const PlaneShape &ps, const void *planes, u8 *g, const u32 *reserved, hipStream_t s);

// State hash of the grid into the partial sums; g holds the bytes of reserved cells.
hipError_t launch_plane_hash(const PlaneShape &ps, const void *planes, const u8 *g, const u32 *reserved, u64 *parts,
                             hipStream_t s);
hipError_t launch_plane_set(const PlaneShape &ps, void *planes, int x, int y, int z, u8 v, u32 *reserved,
                            hipStream_t s);

}  // namespace fs3d
