// Bit planes: the tick on two bits per cell, 32 blocks per 32-bit operation.
//
// A word holds the categories of 64 consecutive cells of a row in four u32:
//   e0, o0   set where a cell is EMPTY or SAND, for the 32 cells with even / odd x
//   e1, o1   set where it is SAND or FLUID
// 16 bytes per 64 cells; a cell's two bits are its category with the low bit
// inverted, so that an all-zero word is STATIC, as cells outside the grid are
// and as buffer loads out of range read.  The pair of cells (2j, 2j + 1) of a word sits at bit
// 2 (j mod 16) + j / 16 of each u32: a block's variant is two adjacent bits of
// its group's 32-bit word (16 blocks per group), so interleaving the words of
// the two groups under a 64-cell word yields the two variant planes in four
// operations, and a shift by one pair is a shift by two bits with two carries.
//
// Reserved bytes (>= 4) are STATIC here; whoever unpacks keeps their bytes.
// Cells past the end of a row are STATIC.
//
// The block rule is a fixed sequence of boolean operations on these planes.
// Variant v renames ring position k to k ^ v (v = 0: the ring itself; 1, 2, 3:
// the scan orders 1032, 2301, 3210), so two conditional swaps bring every block
// into variant 0's frame and the same two bring it back.  In each step a set of
// source cells S and a set of target cells A are matched: sources in scan order
// 0..3, each taking the first remaining target at k + 1, k + 3, k + 2.  A source
// and a target are never in the same column.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define FS3D_HD __host__ __device__ __forceinline__
#else
#define FS3D_HD inline
#endif

namespace fs3d {
namespace plane {

typedef uint32_t u32;

// {hi, lo} >> s, low word (0 < s < 32)
FS3D_HD u32 funnel(u32 hi, u32 lo, int s) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_alignbit(hi, lo, s);
#else
  return (u32)(((((uint64_t)hi) << 32) | lo) >> s);
#endif
}

// Bytes of {a, b} by selector (0..3 from b, 4..7 from a).
FS3D_HD u32 pick_bytes(u32 a, u32 b, u32 sel) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_perm(a, b, sel);
#else
  const uint64_t v = (((uint64_t)a) << 32) | b;
  u32 r = 0;
  for (int i = 0; i < 4; i++) r |= (u32)((v >> (8 * ((sel >> (8 * i)) & 7))) & 0xFF) << (8 * i);
  return r;
#endif
}

FS3D_HD u32 select_bits(u32 m, u32 a, u32 b) { return (a & m) | (b & ~m); }  // m ? a : b

FS3D_HD u32 mix32(u32 h) {  // MurmurHash3's 32-bit finaliser, as the variant spec uses it
  h ^= h >> 16;
  h *= 0x85EBCA6Bu;
  h ^= h >> 13;
  h *= 0xC2B2AE35u;
  h ^= h >> 16;
  return h;
}

// The (y, z, t) part of a variant group's hash input.
FS3D_HD u32 variant_base(u32 by, u32 bz, u32 t) {
  return by * 0x85EBCA77u + bz * 0xC2B2AE3Du + t * 0x27D4EB2Fu;
}

// Variant planes of the 32 blocks whose right (odd ticks) or only (even ticks)
// pair lies in word `seg` of the row: groups 2 seg and 2 seg + 1.
FS3D_HD void variant_planes(u32 seg, u32 base, u32 &v0, u32 &v1) {
  const u32 g = seg * (2u * 0x9E3779B1u) + base;
  const u32 a = mix32(g), b = mix32(g + 0x9E3779B1u);
  v0 = select_bits(0x55555555u, a, b << 1);
  v1 = select_bits(0x55555555u, a >> 1, b);
}

// The odd cells shifted by one pair: bit j of the result is the odd cell of pair
// j - 1, the left cell of odd-parity block j; prev is the word to the left.
FS3D_HD u32 shift_in(u32 o, u32 prev) { return funnel(o, funnel(o >> 30, prev, 1), 30); }

// The inverse: the odd cell of pair j from bit j + 1; bit 0 of next is the
// neighbour's to the right.
FS3D_HD u32 shift_back(u32 l, u32 next) { return funnel(funnel(next, l << 30, 31), l, 2); }

// Three-input bit operations by truth table: A, B and C stand for the operands.
constexpr u32 A = 0xF0, B = 0xCC, C = 0xAA;
template <u32 TT>
FS3D_HD u32 op3(u32 a, u32 b, u32 c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_bitop3_b32(a, b, c, TT & 0xFFu);
#else
  u32 r = 0;
  for (int i = 0; i < 8; i++)
    if ((TT >> i) & 1u) r |= ((i & 4) ? a : ~a) & ((i & 2) ? b : ~b) & ((i & 1) ? c : ~c);
  return r;
#endif
}
constexpr u32 kSelect = (A & B) | (~A & C);  // a ? b : c

// Pins values to this point of the program.  The rule is a few hundred operations
// with little order among them; left alone, the compiler's scheduling keeps many
// more values live than the order written here needs (pair kernel of 2 row quads:
// 177 registers without pins, 151 with two, three waves per SIMD instead of two, for
// 1 % more instructions; a pin after every step: 140, for 4 % more).
template <int N>
FS3D_HD void pin(u32 (&x)[N]) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int i = 0; i < N; i++) asm volatile("" : "+v"(x[i]));
#endif
}

// Matches sources s[0..3] with targets a[0..3]; what remains unmatched stays in
// s and a.  With WALL, the blocks of w only match columns of the same x (ring
// positions k and 3 - k, which the variant's renaming keeps paired).  With UP,
// up[j] receives f[t] of the target source j took.
template <bool WALL, bool UP>
FS3D_HD void match(u32 (&s)[4], u32 (&a)[4], u32 w, const u32 *f, u32 *up) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    u32 r = s[j], g = 0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int t = (j + (i == 0 ? 1 : i == 1 ? 3 : 2)) & 3;
      const u32 at = a[t];
      const bool walled = WALL && t != (j ^ 3);
      if (UP) {
        const u32 m = op3<(A & B & C)>(r, at, walled ? f[4 + t] : f[t]);
        g = i == 0 ? m : g | m;
      }
      a[t] = walled ? op3<(A & ~(B & ~C))>(at, r, w) : at & ~r;
      r = walled ? op3<(A & ~(B & ~C))>(r, at, w) : r & ~at;
    }
    s[j] = r;
    if (UP) up[j] = g;
  }
}

// One tick of 32 blocks: lo / hi[layer][ring position] (0 bottom, 1 top layer;
// ring positions 0..3 = (x, y) (0,0), (1,0), (1,1), (0,1)).  Returns the blocks
// that changed.  The operations are spelled out three operands at a time: left
// to the compiler, the expressions are re-associated across the matches, which
// costs operations (the WALL form: 70) and registers.
template <bool WALL>
FS3D_HD u32 block_rule(u32 (&lo)[2][4], u32 (&hi)[2][4], u32 v0, u32 v1, u32 w) {
  auto cswap = [](u32 m, u32 &x, u32 &y) {
    const u32 p = op3<kSelect>(m, y, x), q = op3<kSelect>(m, x, y);
    x = p;
    y = q;
  };
  auto rename = [&](u32 (&x)[4]) {
    cswap(v0, x[0], x[1]);
    cswap(v0, x[2], x[3]);
    cswap(v1, x[0], x[2]);
    cswap(v1, x[1], x[3]);
  };
#pragma unroll
  for (int l = 0; l < 2; l++) {
    rename(lo[l]);
    rename(hi[l]);
  }
  u32 chg = 0;
  // fall: SAND or FLUID over EMPTY, SAND over FLUID; both cells have then moved
  u32 s[4], fl[4], te[4], a[4], fluid[8];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const u32 lb = lo[0][k], hb = hi[0][k], lt = lo[1][k], ht = hi[1][k];
    const u32 f = ht & op3<(A & ~B) | (C & ~A & B)>(lb, hb, lt);
    lo[0][k] = op3<kSelect>(f, lt, lb);
    hi[0][k] = op3<kSelect>(f, ht, hb);
    lo[1][k] = op3<kSelect>(f, lb, lt);
    hi[1][k] = op3<kSelect>(f, hb, ht);
    s[k] = op3<(A & B & ~C)>(ht, lt, f);    // top SAND
    fl[k] = op3<(A & ~B & ~C)>(ht, lt, f);  // top FLUID
    te[k] = op3<(~A & B & ~C)>(ht, lt, f);  // top EMPTY
    a[k] = op3<((A ^ B) & ~C)>(lb, hb, f);  // bottom EMPTY or FLUID
    fluid[k] = hi[0][k];
    if (WALL) fluid[4 + k] = hi[0][k] & ~w;
    chg = k ? chg | f : f;
  }
  // slide: top SAND with a bottom EMPTY or FLUID cell, whose content goes up
  u32 s0[4], a0[4], up[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    s0[k] = s[k];
    a0[k] = a[k];
  }
  pin(lo[0]), pin(lo[1]), pin(hi[0]), pin(hi[1]);
  match<WALL, true>(s, a, w, fluid, up);
  u32 e[4], fb[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const u32 slid = s0[k] & ~s[k], sand = a0[k] & ~a[k];
    hi[1][k] = op3<((A & ~B) | C)>(hi[1][k], slid, up[k]);
    lo[1][k] = lo[1][k] & ~up[k];
    e[k] = a[k] & ~hi[0][k];  // bottom EMPTY
    fb[k] = a[k] & hi[0][k];  // bottom FLUID
    lo[0][k] = lo[0][k] | sand;
    hi[0][k] = hi[0][k] | sand;
    chg = chg | sand;
  }
  // topple: top FLUID with a bottom EMPTY cell; spread: FLUID with an EMPTY cell
  // of its layer, the bottom layer's targets being what topple left
  u32 e0[4], fb0[4], fl0[4], te0[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    e0[k] = e[k];
    fb0[k] = fb[k];
    fl0[k] = fl[k];
    te0[k] = te[k];
  }
  pin(lo[0]), pin(lo[1]), pin(hi[0]), pin(hi[1]);
  match<WALL, false>(fl, e, w, nullptr, nullptr);
  match<WALL, false>(fb, e, w, nullptr, nullptr);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const u32 fill = e0[k] & ~e[k], gone = fb0[k] & ~fb[k];
    lo[0][k] = op3<((A & ~B) | C)>(lo[0][k], fill, gone);
    hi[0][k] = op3<((A & ~B) | C)>(hi[0][k], gone, fill);
    chg = chg | fill;
  }
  match<WALL, false>(fl, te, w, nullptr, nullptr);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const u32 left = fl0[k] & ~fl[k], in = te0[k] & ~te[k];
    lo[1][k] = op3<((A & ~B) | C)>(lo[1][k], in, left);
    hi[1][k] = op3<((A & ~B) | C)>(hi[1][k], left, in);
    chg = chg | in;
  }
#pragma unroll
  for (int l = 0; l < 2; l++) {
    rename(lo[l]);
    rename(hi[l]);
  }
  return chg;
}

// 64 bytes of a row (values 0..3) into a word: w = {e0, o0, e1, o1}.
// d holds the values with the low bit inverted; so does unpack_word's result.
// Dword k = (j4 j3 j2 j1) of the row holds pairs 2k and 2k + 1 (j0); four dwords
// share a byte's four 2-bit fields, two such words its low and high planes, and
// one exchange of index bits (positions 6 apart) leaves bit (j3 j2 j1 j0 j4).
FS3D_HD void pack_word(const u32 (&d)[16], u32 (&w)[4]) {
  u32 lo[2], hi[2];
#pragma unroll
  for (int j3 = 0; j3 < 2; j3++) {
    u32 t[2];
#pragma unroll
    for (int j4 = 0; j4 < 2; j4++) {
      const int k = 8 * j4 + 4 * j3;
      t[j4] = d[k] | (d[k + 2] << 2) | (d[k + 1] << 4) | (d[k + 3] << 6);
    }
    lo[j3] = select_bits(0x55555555u, t[0], t[1] << 1);
    hi[j3] = select_bits(0x55555555u, t[0] >> 1, t[1]);
  }
  w[0] = pick_bytes(lo[1], lo[0], 0x06040200u);
  w[1] = pick_bytes(lo[1], lo[0], 0x07050301u);
  w[2] = pick_bytes(hi[1], hi[0], 0x06040200u);
  w[3] = pick_bytes(hi[1], hi[0], 0x07050301u);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const u32 x = (w[i] ^ (w[i] >> 6)) & 0x00CC00CCu;
    w[i] ^= x ^ (x << 6);
  }
}

// The inverse of pack_word.
FS3D_HD void unpack_word(const u32 (&w_in)[4], u32 (&d)[16]) {
  u32 w[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const u32 x = (w_in[i] ^ (w_in[i] >> 6)) & 0x00CC00CCu;
    w[i] = w_in[i] ^ x ^ (x << 6);
  }
  u32 lo[2], hi[2];
  lo[0] = pick_bytes(w[1], w[0], 0x05010400u);
  lo[1] = pick_bytes(w[1], w[0], 0x07030602u);
  hi[0] = pick_bytes(w[3], w[2], 0x05010400u);
  hi[1] = pick_bytes(w[3], w[2], 0x07030602u);
#pragma unroll
  for (int j3 = 0; j3 < 2; j3++) {
    u32 t[2];
    t[0] = select_bits(0x55555555u, lo[j3], hi[j3] << 1);
    t[1] = select_bits(0x55555555u, lo[j3] >> 1, hi[j3]);
#pragma unroll
    for (int j4 = 0; j4 < 2; j4++) {
      const int k = 8 * j4 + 4 * j3;
      d[k] = t[j4] & 0x03030303u;
      d[k + 2] = (t[j4] >> 2) & 0x03030303u;
      d[k + 1] = (t[j4] >> 4) & 0x03030303u;
      d[k + 3] = (t[j4] >> 6) & 0x03030303u;
    }
  }
}

// Bit of pair j within a word's u32.
FS3D_HD int pair_bit(int j) { return 2 * (j & 15) + (j >> 4); }

}  // namespace plane
}  // namespace fs3d
