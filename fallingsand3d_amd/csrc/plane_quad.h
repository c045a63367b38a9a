// Device pieces shared by the bit-plane kernels: a row quad's update in registers,
// plane grids as buffers, and words to and from bytes.
#pragma once

#include "plane.h"
#include "plane_core.h"
#include "tick_core.h"

namespace fs3d {
namespace planedev {

using namespace plane;
using tickcore::dmix64;
using tickcore::u32x4;
using tickcore::u32x4_u;
using tickcore::wave_sum_u64;

// A plane grid as a buffer: loads out of range read 0 (STATIC), stores out of
// range are dropped, so rows outside the grid need no branches.
constexpr u32 kOutside = 0xFFFFFFF0u;  // an offset beyond every grid

struct Planes {
  __amdgpu_buffer_rsrc_t rsrc;
  u32 last;  // offset of the last word
  __device__ __forceinline__ Planes(const void *p, u32 bytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000)), last(bytes - 16u) {}
  // A lane's offset plus a wave-uniform one; 0 beyond the buffer.  The range check
  // compares `off` with the buffer's size minus the scalar offset, which must not
  // exceed it (`last` is a word of zeros, like everything beyond).
  __device__ __forceinline__ u32x4 load(u32 off, u32 uniform = 0) const {
    return __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)off, (int)(uniform < last ? uniform : last), 0);
  }
  // Stored without a scalar offset: with one, a vector instruction that
  // rewrites the data's registers right behind a 16-byte store has changed what was
  // stored, and the compiler keeps the two apart only for stores that have none.
  __device__ __forceinline__ void store(u32 off, u32x4 v) const {
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (int)off, 0, 0);
  }
  __device__ __forceinline__ void store(bool on, u32 off, u32x4 v) const { store(on ? off : kOutside, v); }
};

__device__ __forceinline__ u32 from_lane(int addr, u32 v) { return (u32)__builtin_amdgcn_ds_bpermute(addr, (int)v); }

// The block rule on a row quad at even parity: every block lies within the words.
__device__ __forceinline__ u32 quad_even(u32x4 (&r)[4], u32 seg, u32 base) {
  u32 lo[2][4], hi[2][4], v0, v1;
  variant_planes(seg, base, v0, v1);
#pragma unroll
  for (int l = 0; l < 2; l++) {
    const u32x4 p = r[2 * l], q = r[2 * l + 1];
    lo[l][0] = p.x, lo[l][1] = p.y, lo[l][2] = q.y, lo[l][3] = q.x;
    hi[l][0] = p.z, hi[l][1] = p.w, hi[l][2] = q.w, hi[l][3] = q.z;
  }
  const u32 chg = block_rule<false>(lo, hi, v0, v1, 0u);
#pragma unroll
  for (int l = 0; l < 2; l++) {
    r[2 * l] = u32x4{lo[l][0], lo[l][1], hi[l][0], hi[l][1]};
    r[2 * l + 1] = u32x4{lo[l][3], lo[l][2], hi[l][3], hi[l][2]};
  }
  return chg;
}

// At odd parity: the left cells of a word's blocks are the odd cells one pair to
// the left, the first one from the word before (lane address `prev`); afterwards
// each odd cell comes back from the block to its right (lane address `next`).
// A row's words form a ring.  Where the last word is full (WALL), block 0 of
// word 0 joins two half blocks, the row's last odd column and its first even
// one, with a wall between them (w); otherwise the last odd cell is STATIC
// padding and block 0 is an ordinary block beside it.
template <bool WALL>
__device__ __forceinline__ u32 quad_odd(u32x4 (&r)[4], u32 seg, u32 base, int prev, int next, u32 w) {
  u32 lo[2][4], hi[2][4], v0, v1;
  variant_planes(seg, base, v0, v1);
#pragma unroll
  for (int l = 0; l < 2; l++) {
    const u32x4 p = r[2 * l], q = r[2 * l + 1];
    lo[l][0] = shift_in(p.y, from_lane(prev, p.y));
    lo[l][1] = p.x;
    lo[l][2] = q.x;
    lo[l][3] = shift_in(q.y, from_lane(prev, q.y));
    hi[l][0] = shift_in(p.w, from_lane(prev, p.w));
    hi[l][1] = p.z;
    hi[l][2] = q.z;
    hi[l][3] = shift_in(q.w, from_lane(prev, q.w));
  }
  const u32 chg = block_rule<WALL>(lo, hi, v0, v1, w);
#pragma unroll
  for (int l = 0; l < 2; l++) {
    r[2 * l] = u32x4{lo[l][1], shift_back(lo[l][0], from_lane(next, lo[l][0])), hi[l][1],
                     shift_back(hi[l][0], from_lane(next, hi[l][0]))};
    r[2 * l + 1] = u32x4{lo[l][2], shift_back(lo[l][3], from_lane(next, lo[l][3])), hi[l][2],
                         shift_back(hi[l][3], from_lane(next, hi[l][3]))};
  }
  return chg;
}

// 64 bytes of a row (loaded whole: up to 63 bytes past its end) as a word; cells
// from m on are STATIC, reserved bytes too and set *reserved.
__device__ __forceinline__ u32x4 word_from_bytes(const u8 *p, int m, bool *reserved) {
  u32 d[16];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const u32x4 v = *reinterpret_cast<const u32x4_u *>(p + 16 * c);
    d[4 * c] = v.x, d[4 * c + 1] = v.y, d[4 * c + 2] = v.z, d[4 * c + 3] = v.w;
  }
  if (m < 64)
#pragma unroll
    for (int k = 0; k < 16; k++) d[k] = tickcore::keep_bytes(d[k], m - 4 * k);
  u32 res = 0;
#pragma unroll
  for (int k = 0; k < 16; k++) res |= d[k];
  if (__any((res & 0xFCFCFCFCu) != 0)) {
    if ((res & 0xFCFCFCFCu) != 0) *reserved = true;
#pragma unroll
    for (int k = 0; k < 16; k++) d[k] = tickcore::to_codes(d[k], tickcore::reserved_mask(d[k]));
  }
#pragma unroll
  for (int k = 0; k < 16; k++) d[k] ^= 0x01010101u;
  u32 w[4];
  pack_word(d, w);
  return u32x4{w[0], w[1], w[2], w[3]};
}

// Sixteen cells of a word: quarter q holds cells 16 q .. 16 q + 15.
__device__ __forceinline__ void unpack_quarter(const u32x4 &v, int q, u32 (&d)[4]) {
  u32 w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const u32 x = (w[i] ^ (w[i] >> 6)) & 0x00CC00CCu;
    w[i] ^= x ^ (x << 6);
  }
  const u32 sel = (q & 1) ? 0x07030602u : 0x05010400u;
  const u32 lo = pick_bytes(w[1], w[0], sel), hi = pick_bytes(w[3], w[2], sel);
  const u32 t = ((q & 2) ? select_bits(0x55555555u, lo >> 1, hi) : select_bits(0x55555555u, lo, hi << 1)) ^ 0x55555555u;
  d[0] = t & 0x03030303u;
  d[2] = (t >> 2) & 0x03030303u;
  d[1] = (t >> 4) & 0x03030303u;
  d[3] = (t >> 6) & 0x03030303u;
}

// Stores a quarter's m (<= 16) cells at p; with keep, bytes >= 4 already there stay.
__device__ __forceinline__ void store_quarter(u8 *p, int m, u32 (&d)[4], bool keep) {
  if (keep) {
    const u32x4 b = *reinterpret_cast<const u32x4_u *>(p);
    const u32 bb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const u32 rm = tickcore::reserved_mask(bb[k]);
      d[k] = (bb[k] & rm) | (d[k] & ~rm);
    }
  }
  if (m == 16) {
    *reinterpret_cast<u32x4_u *>(p) = u32x4{d[0], d[1], d[2], d[3]};
  } else {
#pragma unroll
    for (int k = 0; k < 16; k++)
      if (k < m) p[k] = (u8)(d[k >> 2] >> (8 * (k & 3)));
  }
}

// A quarter's share of the state hash: its first m cells, the first of them cell
// i0 of the grid; with `bytes`, STATIC cells are read from there (the quarter's
// bytes), where reserved ones keep their values.
// (`cells`: the ones to mix, a bit each.)
__device__ __forceinline__ u64 hash_quarter(const u32x4 &v, int q, int m, u64 i0, const u8 *bytes,
                                            u32 cells = 0xFFFFu) {
  // pairs 8q .. 8q + 7 sit 2 bits apart: even cells in place, odd ones beside them
  const int sh = 16 * (q & 1) + (q >> 1);
  const u32 x = ((v.x >> sh) & 0x5555u) | (((v.y >> sh) & 0x5555u) << 1);
  const u32 h = ((v.z >> sh) & 0x5555u) | (((v.w >> sh) & 0x5555u) << 1);
  u32 ne = (~x | h) & cells & (m >= 16 ? 0xFFFFu : m > 0 ? (1u << m) - 1u : 0u);
  u64 acc = 0;
  while (ne) {
    const int k = __builtin_ctz(ne);
    ne &= ne - 1u;
    u32 val = (((h >> k) & 1u) << 1) | (~(x >> k) & 1u);
    if (bytes && val == FS3D_STATIC) {
      const u32 b = bytes[k];
      val = b >= 4u ? b : val;
    }
    acc += dmix64(((i0 + (u64)k) << 8) | val);
  }
  return acc;
}

}  // namespace planedev
}  // namespace fs3d
