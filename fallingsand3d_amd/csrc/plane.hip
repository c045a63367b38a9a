// Bit-plane kernels: packing, unpacking, single ticks, pairs of ticks and the
// state hash on two bits per cell (plane_core.h has the layout and the rule).
//
// A plane grid is rows of lr = ceil(nx / 64) words of 16 bytes, v[z][y][word], with
// a row of zeros (STATIC) before every layer's first row and a layer of them at
// either end: the rows around the grid that its border blocks read are memory like
// any other, and a quad's four loads differ by uniform offsets.  One lane holds one
// word of each of a row quad's four rows.
//
// What this replaces: the byte kernels move 2 bytes per voxel-update and gather
// one 8-byte table entry per block (510 vector instructions per 1024 blocks and
// the gathers' latency).  Here a single tick moves 0.5 bytes and takes about 335
// instructions per 2048 blocks, none of them a load, and a pair of ticks moves
// about 0.3 bytes per voxel-update.  Dense ticks on an MI355X, us per tick, byte
// kernels / single plane ticks / plane pairs:
//   512^3            42 / 11.5 / 8.7      (11.7 and 15.4 T voxel-updates/s)
//   1000 x 701 x 603 186 (fused pairs 182) / 34 / 23.5
//   2048^3           3070 (fused pairs 2300) / 770 / 416
// Single ticks are bound by memory (2048^3: 4.3 GB in 770 us, 5.6 TB/s), pairs by
// their instructions (1.3 evaluations per row quad and tick with the halo).
#include "plane_quad.h"
#include "plane_plan.h"

namespace fs3d {
namespace {

using namespace planedev;

constexpr u32 kXcds = 8;  // workgroup i is dispatched to XCD i % 8

__device__ __forceinline__ u64 tick_of(const PlaneArgs &a) { return a.tick_dev ? *a.tick_dev + a.k_off : a.t; }

// A lane's place: word `seg` of strip `unit` (rows, row quads or strips of row
// quads), several units per wave.
struct Lane {
  int unit, seg;
  int prev, next;  // lane addresses of the ring neighbours
  bool in;         // the lane holds a word
  u32 wall;
};

__device__ __forceinline__ Lane lane_of(const PlaneArgs &a, int first_unit, int lane) {
  Lane L;
  const int ul = (int)(((u32)lane * a.lr_magic) >> 16);
  L.seg = lane - ul * a.lr;
  L.unit = first_unit + ul;
  L.in = ul < a.upw;
  const int up = L.seg == 0 ? lane + a.lr - 1 : lane - 1, dn = L.seg == a.lr - 1 ? lane - (a.lr - 1) : lane + 1;
  L.prev = (L.in ? up : lane) * 4;
  L.next = (L.in ? dn : lane) * 4;
  L.wall = L.seg == 0 ? 1u : 0u;
  return L;
}

// A layer's words are contiguous, so a lane's place in the planes is its index in the
// layer; its row, and with it its place in the bytes, takes one multiplication
// (magic = ceil(2^32 / d), exact while the layer's index times d stays below 2^32;
// 0 asks for a division).
__device__ __forceinline__ u32 div_by(u32 i, u32 d, u32 magic) { return magic ? __umulhi(i, magic) : i / d; }

struct LayerArgs {
  int nx, ny, nz, lr;
  u32 magic;  // of the words of a row (or of a tile's eight), times the lanes per word
  u32 words;  // of a layer
  size_t first, stride;  // word 0 of layer 0, words from layer to layer
  bool tiled;
};

// Row and word of a lane's place i in a layer, `per` lanes to a word (sub: which of
// them).  Rows outside the grid (tiles have some) are >= ny.
__device__ __forceinline__ u32 place(const LayerArgs &a, u32 i, u32 per, u32 *seg, u32 *sub) {
  const u32 d = per * (u32)a.lr * (a.tiled ? 8u : 1u);
  const u32 q = div_by(i, d, a.magic), rest = i - q * d;
  *sub = rest % per;
  const u32 w = rest / per;
  *seg = a.tiled ? w >> 3 : w;
  return a.tiled ? 8u * q + (w & 7u) - 8u : q;
}

// First word of a layer.
__device__ __forceinline__ size_t layer_word(const LayerArgs &a, int z) { return a.first + (size_t)z * a.stride; }

// ---- state hash --------------------------------------------------------------------
// Four lanes per word, each mixing its quarter's non-empty cells, or 16 lanes in a
// small grid.  With *reserved, STATIC cells are read from the bytes.  Workgroup
// `block` of gx * gy adds its sum to one of the slots, which start at 0.
//
// Bound by the mixing, about 190 cycles per 64 cells (two 64-bit products at a quarter
// of the rate): 117 us at 512^3 with 35 % of the cells not empty.  In a small grid a
// lane's chain of mixes is what takes the time: a hashed tick of 64^3 takes 4.6 us
// with four lanes per word and 3.6 with 16; of 256 x 120 x 60, where there are waves
// enough, 5.2 and 7.7.
constexpr size_t kSplitHashWords = 1u << 13;  // with 16 lanes per word up to here
struct HashArgs {
  LayerArgs l;
  const u32x4 *in;
  const u8 *g;
  const u32 *reserved;
  u64 *out;  // slots sums, kHashStride apart
  u32 gx, gy, slots;
  int split;  // lanes per quarter (1 or 4)
};

__device__ __forceinline__ void hash_block(const HashArgs &h, u32 block) {
  const LayerArgs &a = h.l;
  const bool bytes = *h.reserved != 0;
  const u32 by = block / h.gx, bx = block - by * h.gx;
  u64 acc = 0;
  const u32 lane = bx * 256u + threadIdx.x;
  const u32 i = h.split == 4 ? lane >> 2 : lane, cells = h.split == 4 ? 0xFu << 4 * (lane & 3u) : 0xFFFFu;
  u32 seg, sub;
  const u32 y = place(a, i, 4, &seg, &sub);
  const int c = (int)(4 * seg + sub);
  const int m = i < 4u * a.words && y < (u32)a.ny ? min(16, a.nx - 16 * c) : 0;
  if (m > 0)
    for (int z = (int)by; z < a.nz; z += (int)h.gy) {
      const u64 i0 = ((u64)z * (u32)a.ny + y) * (u32)a.nx + (u32)(16 * c);
      acc += hash_quarter(h.in[layer_word(a, z) + (i >> 2)], c & 3, m, i0, bytes ? h.g + i0 : nullptr, cells);
    }
  __shared__ u64 wsum[4];
  acc = wave_sum_u64(acc);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const u64 tot = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    if (tot)
      atomicAdd((unsigned long long *)(h.out + (size_t)(block % h.slots) * kHashStride), (unsigned long long)tot);
  }
}

__global__ __launch_bounds__(256) void plane_hash_kernel(HashArgs h) { hash_block(h, blockIdx.x); }

// ---- single tick ----------------------------------------------------------------
// The first hash_blocks workgroups hash the state that the tick reads: a run that is
// hashed after every tick takes one launch per tick instead of three (tick, partial
// sums, their sum): 3.6 us per tick instead of 9.1 at 64^3.
template <bool WALL>
__global__ __launch_bounds__(256) void plane_tick_kernel(PlaneArgs a, HashArgs h, u32 hash_blocks, u32 tx) {
  if (blockIdx.x < hash_blocks) {
    hash_block(h, blockIdx.x);
    return;
  }
  const u32 block = blockIdx.x - hash_blocks, bz = block / tx, bx = block - bz * tx;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const u64 t64 = tick_of(a);
  const u32 t = (u32)t64;
  const int p = (int)(t & 1u);
  const int nyq = (a.ny + p + 1) >> 1, nzq = (a.nz + p + 1) >> 1;
  const int first = ((int)bx * 4 + wv) * a.upw, zq = (int)bz;
  if (__builtin_amdgcn_readfirstlane(first) >= nyq || zq >= nzq) return;
  const Lane L = lane_of(a, first, lane);
  const Planes src(a.src, a.bytes), dst(a.dst, a.bytes);
  const u32 row = (u32)a.lr * 16u, layer = row * (u32)(a.ny + 1);
  const int y0 = 2 * L.unit - p, z0 = 2 * zq - p;
  const bool in = L.in && L.unit < nyq;
  const u32 off = in ? (u32)(z0 + 1) * layer + (u32)(y0 + 1) * row + (u32)L.seg * 16u : kOutside;
  u32x4 r[4];
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = src.load(off, (i & 1 ? row : 0u) + (i >> 1 ? layer : 0u));
  const u32 base = variant_base((u32)L.unit, (u32)zq, t);
  if (p)
    quad_odd<WALL>(r, (u32)L.seg, base, L.prev, L.next, L.wall);
  else
    quad_even(r, (u32)L.seg, base);
#pragma unroll
  for (int l = 0; l < 2; l++)
    if ((unsigned)(z0 + l) < (unsigned)a.nz) {
      dst.store(in && y0 >= 0, off + (l ? layer : 0u), r[2 * l]);
      dst.store(in && y0 + 1 < a.ny, off + row + (l ? layer : 0u), r[2 * l + 1]);
    }
}

// ---- a pair of ticks --------------------------------------------------------------
// Ticks t (odd) and t + 1 in one pass.  A lane owns K even-parity row quads along
// y (a strip, 2K rows) and sweeps z row-quads [Z0, Z1).  Odd row quad i of layer
// pair s covers rows 2 (Y0 + i) - 1 and + 0 and layers 2s - 1 and 2s, so the even
// row quad (Y0 + j, b) takes its four rows from odd quads j and j + 1 of s = b
// (their upper layers) and s = b + 1 (their lower ones).  Everything stays in
// registers: the upper layers of the previous s (top), and the quad before.
//
// A strip's odd quad K is the next strip's quad 0.  With SHARE, it is evaluated by
// the next strip alone, lr lanes on, and its two rows come from there; the wave's
// last strip then only serves the one before (K odd evaluations per K quads and
// layer pair instead of K + 1, on all strips but one).
template <bool WALL, int K, bool SHARE>
__global__ __launch_bounds__(256) void plane_pair_kernel(PlaneArgs a) {
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const u64 t64 = tick_of(a);
  const u32 t = (u32)t64;
  const u32 G = gridDim.x, bid = blockIdx.x;
  const u32 xcd = bid % kXcds, per = G / kXcds, extra = G % kXcds;
  const int tile = (int)(xcd * per + min(xcd, extra) + bid / kXcds) * 4 + wv;
  const int yt = tile % a.ytiles, zr = tile / a.ytiles;
  const int nzq = (a.nz + 1) >> 1;
  const int Z0 = zr * a.zlen, Z1 = min(Z0 + a.zlen, nzq);
  if (Z0 >= nzq) return;
  const Lane L = lane_of(a, yt * (SHARE ? a.upw - 1 : a.upw), lane);
  const int Y0 = L.unit * K;
  const u32 seg = (u32)L.seg;
  const Planes src(a.src, a.bytes), dst(a.dst, a.bytes);
  const u32 row = (u32)a.lr * 16u, layer = row * (u32)(a.ny + 1);
  // row 2 Y0 - 1 of layer 2 Z0 - 1; strips past the last row are bounded by the buffer
  const u32 off = L.in ? (u32)(2 * Z0) * layer + (u32)(2 * Y0) * row + seg * 16u : kOutside;
  const bool owns = L.in && (!SHARE || L.unit < yt * (a.upw - 1) + a.upw - 1);
  const int beyond = (lane + a.lr < 64 ? lane + a.lr : lane) * 4;  // the same word of the next strip
  constexpr int NI = SHARE ? K : K + 1;  // odd quads evaluated per layer pair
  u32x4 top[2 * K];
  u32x4 nx[4];
#pragma unroll
  for (int r = 0; r < 4; r++) nx[r] = src.load(off, (r & 1 ? row : 0u) + (r >> 1 ? layer : 0u));
  u32 base = 0;  // of odd layer 2 s - 1
  for (int s = Z0; s <= Z1; s++, base += 2u * layer) {
    // the even quad (Y0 + j, s - 1) from the rows of the odd quads around it
    auto even = [&](int j, const u32x4 &low0, const u32x4 &low1) {
      if (s == Z0) return;
      u32x4 e[4] = {top[2 * j], top[2 * j + 1], low0, low1};
      quad_even(e, seg, variant_base((u32)(Y0 + j), (u32)(s - 1), t + 1u));
      const u32 b = base - layer;  // layer 2 s - 2
      const bool on0 = owns && 2 * (Y0 + j) < a.ny, on1 = owns && 2 * (Y0 + j) + 1 < a.ny;
      dst.store(on0, off + (b + (u32)(2 * j + 1) * row), e[0]);
      dst.store(on1, off + (b + (u32)(2 * j + 2) * row), e[1]);
      if (2 * s - 1 < a.nz) {
        dst.store(on0, off + (base + (u32)(2 * j + 1) * row), e[2]);
        dst.store(on1, off + (base + (u32)(2 * j + 2) * row), e[3]);
      }
    };
    u32x4 lowp, upp;  // upper row of the odd quad before: its lower and upper layer
    u32x4 low0, up0;  // SHARE: lower row of quad 0
#pragma unroll
    for (int i = 0; i < NI; i++) {
      u32x4 q[4];
#pragma unroll
      for (int r = 0; r < 4; r++) q[r] = nx[r];
      const u32 at = i < NI - 1 ? base + (u32)(2 * i + 2) * row : base + 2u * layer;
#pragma unroll
      for (int r = 0; r < 4; r++) nx[r] = src.load(off, at + (r & 1 ? row : 0u) + (r >> 1 ? layer : 0u));
      // One quad at a time: left alone, the scheduler interleaves the evaluations
      // of several, for which there are no registers.
      __builtin_amdgcn_sched_barrier(0);
      quad_odd<WALL>(q, seg, variant_base((u32)(Y0 + i), (u32)s, t), L.prev, L.next, L.wall);
      __builtin_amdgcn_sched_barrier(0);
      if (i > 0) {
        even(i - 1, lowp, q[0]);
        top[2 * i - 2] = upp;
        top[2 * i - 1] = q[2];
      } else if (SHARE) {
        low0 = q[0];
        up0 = q[2];
      }
      lowp = q[1];
      upp = q[3];
    }
    if constexpr (SHARE) {
      u32x4 l, u;
#pragma unroll
      for (int c = 0; c < 4; c++) {
        l[c] = from_lane(beyond, low0[c]);
        u[c] = from_lane(beyond, up0[c]);
      }
      even(K - 1, lowp, l);
      top[2 * K - 2] = upp;
      top[2 * K - 1] = u;
    }
  }
}

// ---- ticks of the active items only ----------------------------------------------
// An item is one word of a strip of K even-parity row quads over zlen z row-quads
// (a cell of the strip grid).  A pass (a pair of ticks, or one tick at either end of
// a run) leaves an item alone when nothing in it can change: no block of it changed
// during the last tick of either parity (the pass before, and behind a pass of one tick
// the one before that), and neither did a block that reaches over its faces from a
// neighbour.  Whether a block is a fixed point does not depend on its variant, so a
// block that did not change at its parity's last tick and whose cells did not change
// since does not change.  The destination then already holds the item: it is the
// state of two passes ago.
//
// The flags are plane_plan.h's, each flag of all cells in a row, so that the plan's lanes
// read neighbouring words.  A flag may be set without need, never missing.
//
// Sand columns over a pool at 2048^3, where 12 % of the items have work: 145 us per
// pair of ticks (123 us of it instructions).  With planes kept as rows, where the line
// around a word holds 512 cells of one row, the same pass took 280 us; a pass over
// everything takes 820, the byte kernels' packed schedule 2 x 360.

// One thread per cell: which items have work, appended to the list in word order;
// clears the flags that the pass will write, and adds the changes of the pass before to
// the cells' `since`.  (Reading the flags of the pass before that too, for a single tick,
// takes 4 us at 2^30 voxels.)
// A full last word (nx a multiple of 64) has a virtual neighbour, word lr, whose
// lane evaluates the half blocks at the row's end.
__global__ __launch_bounds__(256) void plane_plan_kernel(const u64 *__restrict__ in, const u64 *__restrict__ older,
                                                         u64 *__restrict__ out, u64 *__restrict__ since, int strips,
                                                         int zcells, int lr, int virt, int first, int older_first,
                                                         u32 *list, u32 *count) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int ncell = strips * zcells;
  const int c = (int)blockIdx.x * 256 + (int)threadIdx.x;
  const u64 bits = lr == 64 ? ~0ull : (1ull << lr) - 1ull;
  u64 act = 0;
  int zr = 0, st = 0;
  if (c < ncell) {
    zr = c / strips;
    st = c - zr * strips;
    act = plan_words(in, strips, zcells, st, zr, first);
    if (older) act |= plan_words(older, strips, zcells, st, zr, older_first);
    act &= bits;
    plan_flags(in, out, since, (size_t)c, (size_t)ncell, first);
  }
  const int n = __builtin_popcountll(act) + (virt && ((act >> (lr - 1)) & 1u) ? 1 : 0);
  int incl = n;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(incl, d, 64);
    if (lane >= d) incl += y;
  }
  __shared__ u32 wsum[4], wbase;
  if (lane == 63) wsum[wv] = (u32)incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    const u32 tot = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    wbase = tot ? atomicAdd(count, tot) : 0u;
  }
  __syncthreads();
  u32 at = wbase + (u32)(incl - n);
  for (int i = 0; i < wv; i++) at += wsum[i];
  const u32 code = (u32)c * (u32)(lr + virt);
  while (act) {
    const int s = __builtin_ctzll(act);
    act &= act - 1ull;
    list[at++] = code + (u32)s;
    if (virt && s == lr - 1) list[at++] = code + (u32)lr;
  }
}

enum { kPair = 0, kOdd, kEven };

// A lane per listed item, 62 per wave: lanes 0 and 63 repeat the items before and
// after the wave's own, so that a word's neighbours are in the lanes beside it when
// they have work.  A neighbour that has none is not looked at: the block across the
// edge is a fixed point, so its cells in this item stay as they are, and it does not
// move with STATIC in the neighbour's cells either (what blocks every move with
// those cells there blocks the moves among the others).
template <int MODE, int K>
__global__ __launch_bounds__(256) void plane_list_kernel(PlaneArgs a, const u32 *__restrict__ list, const u32 *count,
                                                         u64 *flags, u32 *next_count, int strips, int ncell, int virt,
                                                         u32 nwaves) {
  const int lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x == 0) *next_count = 0;
  const u32 wave = blockIdx.x * 4 + (u32)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const u32 t = (u32)tick_of(a);
  const u32 n = *count;
  const Planes src(a.src, a.bytes), dst(a.dst, a.bytes);
  const u32 tile = (u32)a.lr * 128u, layer = tile * (u32)((a.ny + 9) / 8 + 1);
  const int m = a.zlen;
  const int prev = (lane ? lane - 1 : 0) * 4, next = (lane < 63 ? lane + 1 : 63) * 4;
  for (u32 w = wave; w * 62u < n; w += nwaves) {
    const u32 e = w * 62u + (u32)lane - 1u;
    const bool in = e < n;  // (entry -1 is none)
    const u32 code = in ? list[e] : 0xFFFFFF00u;
    const u32 per = (u32)(a.lr + virt), cell = code / per;
    const int seg = (int)(code - cell * per);
    const int zr = (int)(cell / (u32)strips), st = (int)(cell - (u32)zr * (u32)strips);
    const int y0 = st * 2 * K, z0 = zr * 2 * m, by0 = st * K, bz0 = zr * m;
    const u32 cp = from_lane(prev, code), cn = from_lane(next, code);
    const bool has_prev = in && lane > 0 && seg > 0 && cp + 1u == code;
    const bool has_next = in && lane < 63 && seg + 1 < (int)per && cn == code + 1u;
    const bool word = in && seg < a.lr;  // not the virtual word
    const bool mine = word && lane > 0 && lane < 63;
    // rows y0 - 2 + 2 i and the one after, of layer z0 - 1
    u32 off[K + 2];
#pragma unroll
    for (int i = 0; i < K + 2; i++) {
      const u32 pr = (u32)(st * K + i + 3);  // pair of rows: four to a tile
      off[i] = word ? (u32)z0 * layer + (pr >> 2) * tile + (u32)seg * 128u + (pr & 3u) * 32u : kOutside;
    }
    bool on[2 * K];
#pragma unroll
    for (int j = 0; j < 2 * K; j++) on[j] = mine && y0 + j < a.ny;
    const int zleft = a.nz - z0;  // layers of the item inside the grid
    u32 acc[kFlags] = {};
    // odd quad (i, s) in place; returns its changed blocks, bit 31 also standing
    // for the block at the word's right edge
    auto odd = [&](u32x4(&q)[4], int i, int s) {
      u32 lo[2][4], hi[2][4], v0, v1;
      variant_planes((u32)seg, variant_base((u32)(by0 + i), (u32)(bz0 + s), t), v0, v1);
      u32 last = 0;  // last odd cells, kept where no neighbour evaluates their block
#pragma unroll
      for (int r = 0; r < 4; r++) {
        u32 px = from_lane(prev, q[r].y), ph = from_lane(prev, q[r].w);
        px = has_prev ? px : 0u;
        ph = has_prev ? ph : 0u;
        const int l = r >> 1, kl = (r & 1) ? 3 : 0, kr = (r & 1) ? 2 : 1;
        lo[l][kl] = shift_in(q[r].y, px);
        hi[l][kl] = shift_in(q[r].w, ph);
        lo[l][kr] = q[r].x;
        hi[l][kr] = q[r].z;
        last |= (q[r].y >> 31) << r | (q[r].w >> 31) << (4 + r);
      }
      const u32 c = block_rule<false>(lo, hi, v0, v1, 0u);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int l = r >> 1, kl = (r & 1) ? 3 : 0, kr = (r & 1) ? 2 : 1;
        // (read by every lane: a lane left out is not readable by its neighbour)
        u32 nx = from_lane(next, lo[l][kl]), nh = from_lane(next, hi[l][kl]);
        nx = has_next ? nx : last >> r;
        nh = has_next ? nh : last >> (4 + r);
        q[r] = u32x4{lo[l][kr], shift_back(lo[l][kl], nx & 1u), hi[l][kr], shift_back(hi[l][kl], nh & 1u)};
      }
      const u32 cnext = from_lane(next, c);
      return c | (has_next ? cnext << 31 : 0u);
    };
    // (i, s) in quads of the item's rows and layers; quads past the grid hold nothing
    auto note = [&](u32 c, int y, int z, bool yf, bool yl, bool zf, bool zl) {
      c = y0 + y < a.ny && z < zleft ? c : 0u;
      acc[kAny] |= c;
      if (yf) acc[kYFirst] |= c;
      if (yl) acc[kYLast] |= c;
      if (zf) acc[kZFirst] |= c;
      if (zl) acc[kZLast] |= c;
    };
    if constexpr (MODE == kEven) {
      u32 base = layer;  // layer 2 b
#pragma unroll 1
      for (int b = 0; b < m; b++, base += 2u * layer)
#pragma unroll
        for (int j = 0; j < K; j++) {
          u32x4 q[4];
#pragma unroll
          for (int r = 0; r < 4; r++)
            q[r] = src.load(off[j + 1], base + (r & 1 ? 16u : 0u) + (r >> 1 ? layer : 0u));
          const u32 c = quad_even(q, (u32)seg, variant_base((u32)(by0 + j), (u32)(bz0 + b), t));
          note(c, 2 * j, 2 * b, j == 0, j == K - 1, b == 0, b == m - 1);
#pragma unroll
          for (int r = 0; r < 4; r++)
            dst.store(on[2 * j + (r & 1)] && 2 * b + (r >> 1) < zleft,
                      off[j + 1] + (base + (r & 1 ? 16u : 0u) + (r >> 1 ? layer : 0u)), q[r]);
        }
    } else {
      u32x4 top[2 * K], nx[4];
      u32 base = 0;  // layer 2 s - 1
#pragma unroll
      for (int r = 0; r < 4; r++) nx[r] = src.load(off[r & 1], (r & 1 ? 0u : 16u) + (r >> 1 ? layer : 0u));
#pragma unroll 1
      for (int s = 0; s <= m; s++, base += 2u * layer) {
        u32x4 lowp, upp;
#pragma unroll
        for (int i = 0; i <= K; i++) {
          u32x4 q[4];
#pragma unroll
          for (int r = 0; r < 4; r++) q[r] = nx[r];
          const u32 at = i < K ? base : base + 2u * layer;
#pragma unroll
          for (int r = 0; r < 4; r++)
            nx[r] = src.load(off[(i < K ? i + 1 : 0) + (r & 1)], at + (r & 1 ? 0u : 16u) + (r >> 1 ? layer : 0u));
          __builtin_amdgcn_sched_barrier(0);
          const u32 c = odd(q, i, s);
          note(c, 2 * i - 1, 2 * s - 1, i == 0, i == K, s == 0, s == m);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (MODE == kOdd) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const int dy = 2 * i - 1 + (r & 1), dz = 2 * s - 1 + (r >> 1);
              if (dy >= 0 && dy < 2 * K)
                dst.store(on[dy] && (unsigned)dz < (unsigned)min(2 * m, zleft),
                          off[i + (r & 1)] + (base + (r & 1 ? 0u : 16u) + (r >> 1 ? layer : 0u)), q[r]);
            }
          } else {
            if (i > 0) {
              if (s > 0) {
                u32x4 v[4] = {top[2 * i - 2], top[2 * i - 1], lowp, q[0]};
                const u32 c2 = quad_even(v, (u32)seg, variant_base((u32)(by0 + i - 1), (u32)(bz0 + s - 1), t + 1u));
                note(c2, 2 * i - 2, 2 * s - 2, i == 1, i == K, s == 1, s == m);
#pragma unroll
                for (int r = 0; r < 4; r++)
                  dst.store(on[2 * i - 2 + (r & 1)] && 2 * s - 2 + (r >> 1) < zleft,
                            off[i] + (base - layer + (r & 1 ? 16u : 0u) + (r >> 1 ? layer : 0u)), v[r]);
              }
              top[2 * i - 2] = upp;
              top[2 * i - 1] = q[2];
            }
            lowp = q[1];
            upp = q[3];
          }
        }
      }
    }
    // the first lane of each run of neighbouring items ORs the run's flags
    acc[kXFirst] = acc[kAny] & 1u;
    acc[kXLast] = acc[kAny] >> 31;
    acc[kNow] = acc[kAny];
    const u64 starts = __ballot(!has_prev);
    const u64 after = lane < 63 ? starts >> (lane + 1) : 0ull;
    const int len = after ? __builtin_ctzll(after) + 1 : 64 - lane;
    const u64 run = len >= 64 ? ~0ull : (1ull << len) - 1ull;
#pragma unroll
    for (int f = 0; f < kFlags; f++) {
      const u64 b = __ballot(mine && acc[f] != 0u);
      const u64 bits = ((b >> lane) & run) << (seg & 63);
      if (!has_prev && in && bits)
        atomicOr((unsigned long long *)(flags + (size_t)f * ncell + cell), (unsigned long long)bits);
    }
  }
}

// ---- bytes <-> planes --------------------------------------------------------------
// One lane per word: 64 bytes of a row.  *reserved is set when a byte >= 4 is seen
// (the planes hold STATIC for it).
__global__ __launch_bounds__(256) void plane_pack_kernel(const u8 *g, u32x4 *out, LayerArgs a, u32 *reserved) {
  bool any = false;
  const u32 i = blockIdx.x * 256u + threadIdx.x;
  u32 seg, sub;
  u32 y = place(a, i, 1, &seg, &sub);
  const bool in = i < a.words && y < (u32)a.ny;
  const int x0 = in ? (int)seg * 64 : 0;
  y = in ? y : 0u;
  for (int z = (int)blockIdx.y; z < a.nz; z += (int)gridDim.y) {
    // loads may run up to 63 bytes past the last row, into the guard bytes
    const u32x4 v = word_from_bytes(g + ((size_t)z * (u32)a.ny + y) * (u32)a.nx + (u32)x0, min(64, a.nx - x0), &any);
    if (in) out[layer_word(a, z) + i] = v;
  }
  if (__any(any) && (threadIdx.x & 63) == 0) *reserved = 1u;
}

// Packing and the tick after it in one pass, for an even tick t, whose blocks lie in
// their words: the planes are written once instead of written, read and written.  A
// lane packs and ticks one word of m row quads along z.  flags (of items, 0 before; or
// nullptr): kNow where a cell changed, kAny where one is sand or fluid and so may; the
// next pass then leaves items alone that it did not write, so what cannot move goes to
// its destination (a.src) too.
//
// Bound by memory: 2048^3 in 2.30 ms, 12.9 GB at 5.6 TB/s (packing alone takes 2.15, the
// tick after it took 1.95, and the pair after that 2.3 where it now takes 0.13).  Lines
// of tiles are written whole by a wave: with the tiles one row further up, so that each
// wave wrote 7/8 of its lines, it took 4.2.
template <bool TILED>
__global__ __launch_bounds__(256) void plane_pack_even_kernel(const u8 *g, int nx, PlaneArgs a, int m, int strips,
                                                              int ncell, u64 *flags, u32 *reserved) {
  const u32 t = (u32)tick_of(a);
  const Planes dst(a.dst, a.bytes), other(a.src, a.bytes);
  const int nzq = (a.nz + 1) >> 1;
  const u32 i = blockIdx.x * 256u + threadIdx.x, lr = (u32)a.lr;
  // rows: words along a row; tiles: a tile's four strips of a word, so that its lines
  // are written whole
  const u32 over = i / (TILED ? 4u * lr : lr), rest = i - over * (TILED ? 4u * lr : lr);
  const u32 st = TILED ? 4u * over + (rest & 3u) : over, seg = TILED ? rest >> 2 : rest;
  const u32 tiles = (u32)(a.ny + 9) / 8u + 1u;
  const int y0 = 2 * (int)st;
  const bool in = y0 < a.ny;
  bool any = false;
  for (int zr = (int)blockIdx.y; zr * m < nzq; zr += (int)gridDim.y) {
    u32 acc = 0, mobile = 0;
    for (int zq = zr * m; zq < min((zr + 1) * m, nzq); zq++) {
      u32x4 q[4];
      u32 off[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int y = y0 + (r & 1), z = 2 * zq + (r >> 1);
        const bool ok = in && y < a.ny && z < a.nz;
        const u32 row = (u32)(y + (TILED ? 8 : 1));
        const u32 word = TILED ? (((u32)(z + 1) * tiles + (row >> 3)) * lr + seg) * 8u + (row & 7u)
                               : ((u32)(z + 1) * (u32)(a.ny + 1) + row) * lr + seg;
        off[r] = ok ? word * 16u : kOutside;
        q[r] = word_from_bytes(ok ? g + ((size_t)z * (u32)a.ny + (u32)y) * (u32)nx + 64u * seg : g,
                               ok ? min(64, nx - 64 * (int)seg) : 0, &any);
      }
      acc |= quad_even(q, seg, variant_base(st, (u32)zq, t));
      u32 high = 0;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        high |= q[r].z | q[r].w;
        dst.store(off[r], q[r]);
      }
      mobile |= high;
      if (flags)  // an item in which nothing can move may be left alone by the next pass
#pragma unroll
        for (int r = 0; r < 4; r++) other.store(high == 0, off[r], q[r]);
    }
    if (flags && in) {
      unsigned long long *f = (unsigned long long *)(flags + ((size_t)zr * (u32)strips + st));
      if (acc) atomicOr(f + (size_t)kNow * ncell, 1ull << seg);
      if (mobile) atomicOr(f + (size_t)kAny * ncell, 1ull << seg);
    }
  }
  if (__any(any) && (threadIdx.x & 63) == 0) *reserved = 1u;
}

// Planes to bytes, four lanes per word so that a wave stores 1 KiB in a row.
__global__ __launch_bounds__(256) void plane_unpack_kernel(const u32x4 *in, u8 *g, LayerArgs a, const u32 *reserved) {
  const bool keep = *reserved != 0;
  const u32 i = blockIdx.x * 256u + threadIdx.x;
  u32 seg, sub;
  const u32 y = place(a, i, 4, &seg, &sub);
  const int c = (int)(4 * seg + sub), m = min(16, a.nx - 16 * c);
  if (i >= 4u * a.words || y >= (u32)a.ny || m <= 0) return;
  for (int z = (int)blockIdx.y; z < a.nz; z += (int)gridDim.y) {
    u32 d[4];
    unpack_quarter(in[layer_word(a, z) + (i >> 2)], c & 3, d);
    // reserved cells hold their bytes (they never move)
    store_quarter(g + ((size_t)z * (u32)a.ny + y) * (u32)a.nx + (u32)(16 * c), m, d, keep);
  }
}

// The rows around the grid: the layers before the first and after the last, and the
// row between every two layers; in tiles, the first and what is behind the last row.
__global__ __launch_bounds__(256) void plane_pad_kernel(u32x4 *p, int ny, int nz, int lr) {
  const size_t end = (size_t)(ny + 1) * (u32)lr, mid = (size_t)nz * (u32)lr, n = 2 * end + mid + (u32)lr;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    size_t w;
    if (i < end) {
      w = i;
    } else if (i < end + mid) {
      const size_t k = i - end, z = k / (u32)lr;
      w = (z + 1) * end + (k - z * (u32)lr);
    } else {
      w = (size_t)(nz + 1) * end + (i - end - mid);
    }
    p[w] = u32x4{0u, 0u, 0u, 0u};
  }
}

__global__ __launch_bounds__(256) void plane_pad_tiles_kernel(u32x4 *p, int ny, int nz, int lr, int tiles) {
  const u32 tile = 8u * (u32)lr, layer = tile * (u32)tiles, last = (u32)(ny + 8) / 8u;  // the tile of row ny
  const u32 mid = tile * (1u + (u32)tiles - last);  // words of a layer of the grid that may be outside it
  const u64 n = 2 * (u64)layer + (u64)mid * (u32)nz;
  for (u64 i = (u64)blockIdx.x * 256 + threadIdx.x; i < n; i += (u64)gridDim.x * 256) {
    u64 w = i;
    if (i >= layer && i < layer + (u64)mid * (u32)nz) {
      const u32 z = (u32)((i - layer) / mid), k = (u32)((i - layer) - (u64)z * mid);
      const u32 t = k < tile ? 0u : last - 1u + k / tile;
      if (t >= last && t * 8u + (k & 7u) < (u32)(ny + 8)) continue;  // (a tile's words: word, row)
      w = (u64)(z + 1u) * layer + (u64)t * tile + k % tile;
    } else if (i >= layer) {
      w = (u64)(nz + 1) * layer + (i - layer - (u64)mid * (u32)nz);
    }
    p[w] = u32x4{0u, 0u, 0u, 0u};
  }
}

// Unpacks the items changed since the bytes were last written: a wave per cell of
// the strip grid, 16 words of a row at a time.  With dirty, the renderer's bricks that
// they lie in are marked: reading the bricks of what moved in ten ticks of 1024^3 sand
// columns takes 76 us, reading all of them 204.
__global__ __launch_bounds__(256) void plane_unpack_cells_kernel(const u32x4 *in, u8 *g, int nx, int ny, int nz, int lr,
                                                                 u32 layer, int strips, int ncell, int rows, int layers,
                                                                 const u64 *flags, u64 *since, const u32 *reserved,
                                                                 u64 *dirty) {
  const int lane = threadIdx.x & 63;
  const int c = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (c >= ncell) return;
  const u64 bits = since[c] | flags[(size_t)kNow * ncell + c];
  if (bits == 0) return;
  const bool keep = *reserved != 0;
  const int zr = c / strips, st = c - zr * strips;
  const int q = lane & 3;
  for (int s0 = 0; s0 < lr; s0 += 16) {
    if (((bits >> s0) & 0xFFFFull) == 0) continue;
    const int seg = s0 + (lane >> 2);
    const int x0 = 64 * seg + 16 * q, m = min(16, nx - x0);
    if (seg >= lr || !((bits >> seg) & 1ull) || m <= 0) continue;
    for (int dz = 0; dz < layers; dz++) {
      const int z = zr * layers + dz;
      if (z >= nz) break;
#pragma unroll 4
      for (int dy = 0; dy < rows; dy++) {
        const int y = st * rows + dy;
        if (y < ny) {
          u32 d[4];
          const u32 row = (u32)(y + 8);  // (tiled planes)
          unpack_quarter(in[(size_t)(z + 1) * layer + ((row >> 3) * (u32)lr + (u32)seg) * 8u + (row & 7u)], q, d);
          store_quarter(g + ((size_t)z * (u32)ny + (u32)y) * (u32)nx + (u32)x0, m, d, keep);
        }
      }
    }
  }
  if (lane == 0) since[c] = 0;
  if (dirty) {  // the 8^3 bricks of the changed words: a word's eight are a byte of their row
    const int bwords = (nx + 511) / 512, bny = (ny + 7) / 8;
    const int j = lane % bwords, z = zr * layers + 8 * (lane / bwords);
    if (z < min((zr + 1) * layers, nz)) {
      u64 m = (bits >> (8 * j)) & 0xFFull;
      m = (m | m << 28) & 0x0000000F0000000Full;
      m = (m | m << 14) & 0x0003000300030003ull;
      m = (m | m << 7) & 0x0101010101010101ull;
      if (m) atomicOr((unsigned long long *)(dirty + ((size_t)(z / 8) * bny + st * rows / 8) * bwords + j), m * 0xFFull);
    }
  }
}

}  // namespace

static void fill_args(PlaneArgs &a, const PlaneShape &ps) {
  a.ny = ps.ny;
  a.nz = ps.nz;
  a.lr = ps.lr;
  a.bytes = (u32)(plane_words(ps) * 16);
  a.upw = 64 / ps.lr;
  a.lr_magic = (65536u + (u32)ps.lr - 1u) / (u32)ps.lr;
}

// per: lanes per word.  Layers per lane: enough blocks for the chip, few enough that
// the row's division and a hash's reduction are shared by several layers.
static LayerArgs layer_args(const PlaneShape &ps, int per, dim3 *grid) {
  const u64 rows = ps.tiled ? (u64)plane_tiles(ps) : (u64)ps.ny;
  const u64 d = (u64)per * (u64)ps.lr * (ps.tiled ? 8 : 1), n = d * rows;
  LayerArgs a{ps.nx, ps.ny, ps.nz, ps.lr, 0, (u32)(n / (u64)per), plane_word(ps, 0, ps.tiled ? -8 : 0, 0),
              plane_word(ps, 0, 0, 1) - plane_word(ps, 0, 0, 0), ps.tiled};
  if (n * d < (1ull << 32) && d > 1) a.magic = (u32)(((1ull << 32) + d - 1) / d);
  const unsigned gx = (unsigned)((n + 255) / 256);
  const unsigned gy = (unsigned)std::min<u64>((u64)std::min(ps.nz, 65535), std::max<u64>(1, 16384 / std::max(gx, 1u)));
  *grid = dim3(gx, gy);
  return a;
}

static HashArgs hash_args(const PlaneShape &ps, const PlaneHash &ph, const void *planes) {
  dim3 grid;
  HashArgs h{};
  h.l = layer_args(ps, 4, &grid);
  h.in = static_cast<const u32x4 *>(planes);
  h.g = ph.g;
  h.reserved = ph.reserved;
  h.gx = grid.x;
  h.gy = grid.y;
  const bool direct = plane_hash_direct(ps);
  h.split = plane_words(ps) <= kSplitHashWords ? 4 : 1;
  if (h.split == 4) h.gx = (unsigned)(((size_t)16 * h.l.words + 255) / 256);
  h.out = direct ? ph.out : ph.parts;
  h.slots = direct ? 1 : kHashParts;
  return h;
}

hipError_t launch_plane_tick(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             const PlaneHash *hash, hipStream_t s) {
  PlaneArgs a{};
  fill_args(a, ps);
  a.src = static_cast<const u32x4 *>(src);
  a.dst = static_cast<u32x4 *>(dst);
  a.t = t;
  a.tick_dev = tick_dev;
  a.k_off = k_off;
  const u32 tx = (u32)plane_tick_rows(ps);
  HashArgs h{};
  u32 hb = 0;
  if (hash) {
    h = hash_args(ps, *hash, src);
    hb = h.gx * h.gy;
  }
  const dim3 grid(hb + (u32)plane_tick_blocks(ps));
  if (ps.nx % 64 == 0)
    hipLaunchKernelGGL(plane_tick_kernel<true>, grid, dim3(256), 0, s, a, h, hb, tx);
  else
    hipLaunchKernelGGL(plane_tick_kernel<false>, grid, dim3(256), 0, s, a, h, hb, tx);
  return hipGetLastError();
}

// The launch shape of a pair.  Per SIMD, w resident waves of e evaluations each take
// about e * max(0.87, 0.6 w) us (one wave alone waits for its own loads), so the
// shape that takes the fewest evaluations is not always the fastest: long sweeps
// evaluate fewer halo quads and leave fewer waves.  K = 2 without sharing is the
// shape of rows too long to share (us per tick at 512^3: K = 1 unshared, zlen 2 / 4 /
// 8: 9.7 / 9.1 / 11.3; K = 2, zlen 2 / 4 / 8: 9.5 / 10.9 / 16.8; 2048^3: K = 1, zlen
// 16 415, K = 2, zlen 8 / 16 409 / 416, all bound by memory).
struct PairShape {
  int k, zlen;
  bool share;
};
static PairShape pair_shape(const PlaneShape &ps) {
  const int upw = 64 / ps.lr, nyq = (ps.ny + 1) >> 1, nzq = (ps.nz + 1) >> 1;
  PairShape best{1, 1, false};
  double least = 1e300;
  for (int v = 0; v < 3; v++) {
    const int k = v == 2 ? 2 : 1;
    const bool share = v == 0;
    const int adv = share ? upw - 1 : upw;  // strips per wave
    if (adv < 1) continue;
    const int strips = (nyq + k - 1) / k, yt = (strips + adv - 1) / adv;
    for (int z = 1; z <= 16; z++) {
      const double waves = (double)yt * ((nzq + z - 1) / z), w = waves / 1024.0;
      const double evals = (double)(share ? k : k + 1) * (z + 1) + (double)k * z;
      const double whole = w > 8.0 ? w : (double)(long long)(w + 0.999);  // the last round of few is not full
      const double t = evals * std::max(0.87, 0.6 * whole);
      if (t < least * 0.999) {
        least = t;
        best = PairShape{k, z, share};
      }
    }
  }
  return best;
}

hipError_t launch_plane_pair(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             hipStream_t s) {
  PlaneArgs a{};
  fill_args(a, ps);
  a.src = static_cast<const u32x4 *>(src);
  a.dst = static_cast<u32x4 *>(dst);
  a.t = t;
  a.tick_dev = tick_dev;
  a.k_off = k_off;
  const PairShape p = pair_shape(ps);
  a.zlen = p.zlen;
  const int nyq = (ps.ny + 1) >> 1, nzq = (ps.nz + 1) >> 1;
  const int strips = (nyq + p.k - 1) / p.k, adv = p.share ? a.upw - 1 : a.upw;
  a.ytiles = (strips + adv - 1) / adv;
  const long long waves = (long long)a.ytiles * ((nzq + p.zlen - 1) / p.zlen);
  const dim3 grid((unsigned)((waves + 3) / 4));
  const bool wall = ps.nx % 64 == 0;
  if (p.share) {
    if (wall) hipLaunchKernelGGL((plane_pair_kernel<true, 1, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((plane_pair_kernel<false, 1, true>), grid, dim3(256), 0, s, a);
  } else if (p.k == 1) {
    if (wall) hipLaunchKernelGGL((plane_pair_kernel<true, 1, false>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((plane_pair_kernel<false, 1, false>), grid, dim3(256), 0, s, a);
  } else {
    if (wall) hipLaunchKernelGGL((plane_pair_kernel<true, 2, false>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((plane_pair_kernel<false, 2, false>), grid, dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

// 512 workgroups at most add to one word; each addition takes it 13 ns (16384 at 512^3
// made the hash 210 us instead of 117).
bool plane_hash_direct(const PlaneShape &ps) { return plane_words(ps) <= (1u << 15); }

PlaneCells plane_cells(const PlaneShape &ps) {
  PlaneCells c;
  c.strips = (((ps.ny + 1) >> 1) + kItemQuads - 1) / kItemQuads;
  c.zcells = (((ps.nz + 1) >> 1) + kItemLayers - 1) / kItemLayers;
  c.virt = ps.nx % 64 == 0 ? 1 : 0;
  const size_t n = (size_t)c.strips * (size_t)c.zcells;
  c.flag_words = n * kFlags;
  c.since_words = n;
  c.list_words = n * (size_t)(ps.lr + c.virt);
  return c;
}

int plane_list_blocks_per_cu() {
  int n = 0;
  const hipError_t e =
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, plane_list_kernel<kPair, kItemQuads>, 256, 0);
  return e == hipSuccess && n > 0 ? n : 1;
}

hipError_t launch_plane_list(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             bool pair, int first, const u64 *flags_in, int older_first, const u64 *older,
                             u64 *flags_out, u64 *since, u32 *list, u32 *count, u32 *next_count, u32 nwaves,
                             hipStream_t s) {
  PlaneArgs a{};
  fill_args(a, ps);
  a.src = static_cast<const u32x4 *>(src);
  a.dst = static_cast<u32x4 *>(dst);
  a.t = t;
  a.tick_dev = tick_dev;
  a.k_off = k_off;
  a.zlen = kItemLayers;
  const PlaneCells c = plane_cells(ps);
  const unsigned plan = (unsigned)((c.since_words + 255) / 256);
  hipLaunchKernelGGL(plane_plan_kernel, dim3(plan), dim3(256), 0, s, flags_in, older, flags_out, since, c.strips,
                     c.zcells, ps.lr, c.virt, first, older_first, list, count);
  const dim3 grid(nwaves / 4);
  // the caller's t has the tick's parity, on replays too
  if (pair)
    hipLaunchKernelGGL((plane_list_kernel<kPair, kItemQuads>), grid, dim3(256), 0, s, a, list, count, flags_out,
                       next_count, c.strips, (int)c.since_words, c.virt, nwaves);
  else if (t & 1u)
    hipLaunchKernelGGL((plane_list_kernel<kOdd, kItemQuads>), grid, dim3(256), 0, s, a, list, count, flags_out,
                       next_count, c.strips, (int)c.since_words, c.virt, nwaves);
  else
    hipLaunchKernelGGL((plane_list_kernel<kEven, kItemQuads>), grid, dim3(256), 0, s, a, list, count, flags_out,
                       next_count, c.strips, (int)c.since_words, c.virt, nwaves);
  return hipGetLastError();
}

hipError_t launch_plane_unpack_cells(const PlaneShape &ps, const void *planes, u8 *g, const u64 *flags, u64 *since,
                                     const u32 *reserved, u64 *dirty, hipStream_t s) {
  const PlaneCells c = plane_cells(ps);
  const int ncell = (int)c.since_words;
  hipLaunchKernelGGL(plane_unpack_cells_kernel, dim3((unsigned)((ncell + 3) / 4)), dim3(256), 0, s,
                     static_cast<const u32x4 *>(planes), g, ps.nx, ps.ny, ps.nz, ps.lr,
                     (u32)(plane_tiles(ps) * 8 * ps.lr), c.strips, ncell,
                     2 * kItemQuads, 2 * kItemLayers, flags, since, reserved, dirty);
  return hipGetLastError();
}

hipError_t launch_plane_pad(const PlaneShape &ps, void *planes, hipStream_t s) {
  if (ps.tiled) {
    hipLaunchKernelGGL(plane_pad_tiles_kernel, dim3(2048), dim3(256), 0, s, static_cast<u32x4 *>(planes), ps.ny, ps.nz,
                       ps.lr, plane_tiles(ps));
    return hipGetLastError();
  }
  const size_t n = ((size_t)2 * (u32)(ps.ny + 1) + (u32)ps.nz + 1) * (u32)ps.lr;
  hipLaunchKernelGGL(plane_pad_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096)), dim3(256), 0, s,
                     static_cast<u32x4 *>(planes), ps.ny, ps.nz, ps.lr);
  return hipGetLastError();
}

hipError_t launch_plane_pack(const PlaneShape &ps, const u8 *g, void *planes, u32 *reserved, hipStream_t s) {
  dim3 grid;
  const LayerArgs a = layer_args(ps, 1, &grid);
  hipLaunchKernelGGL(plane_pack_kernel, grid, dim3(256), 0, s, g, static_cast<u32x4 *>(planes), a, reserved);
  return hipGetLastError();
}

hipError_t launch_plane_pack_even(const PlaneShape &ps, const u8 *g, void *planes, u32 *reserved, u64 t,
                                  const u64 *tick_dev, u32 k_off, u64 *flags, void *other, hipStream_t s) {
  PlaneArgs a{};
  fill_args(a, ps);
  a.src = static_cast<const u32x4 *>(flags ? other : planes);
  a.dst = static_cast<u32x4 *>(planes);
  a.t = t;
  a.tick_dev = tick_dev;
  a.k_off = k_off;
  const PlaneCells c = plane_cells(ps);
  if (flags) {
    const hipError_t e = launch_fill_u64(flags, c.flag_words, 0, s);
    if (e != hipSuccess) return e;
  }
  const int nyq = (ps.ny + 1) >> 1, nzq = (ps.nz + 1) >> 1;
  const u32 gx = (u32)(((u64)(ps.tiled ? (nyq + 3) / 4 * 4 : nyq) * (u64)ps.lr + 255) / 256);
  // items' layers, or what keeps the chip busy
  const int m = flags ? kItemLayers : (int)std::min<u64>(8, std::max<u64>(1, (u64)gx * (u64)nzq / 4096));
  const dim3 grid(gx, (unsigned)std::min((nzq + m - 1) / m, 65535));
  if (ps.tiled)
    hipLaunchKernelGGL(plane_pack_even_kernel<true>, grid, dim3(256), 0, s, g, ps.nx, a, m, c.strips, (int)c.since_words, flags, reserved);
  else
    hipLaunchKernelGGL(plane_pack_even_kernel<false>, grid, dim3(256), 0, s, g, ps.nx, a, m, c.strips, (int)c.since_words, flags, reserved);
  return hipGetLastError();
}

hipError_t launch_plane_unpack(const PlaneShape &ps, const void *planes, u8 *g, const u32 *reserved, hipStream_t s) {
  dim3 grid;
  const LayerArgs a = layer_args(ps, 4, &grid);
  hipLaunchKernelGGL(plane_unpack_kernel, grid, dim3(256), 0, s, static_cast<const u32x4 *>(planes), g, a, reserved);
  return hipGetLastError();
}

hipError_t launch_plane_hash(const PlaneShape &ps, const void *planes, const PlaneHash &hash, hipStream_t s) {
  const HashArgs h = hash_args(ps, hash, planes);
  hipLaunchKernelGGL(plane_hash_kernel, dim3(h.gx * h.gy), dim3(256), 0, s, h);
  return hipGetLastError();
}

size_t plane_word(const PlaneShape &ps, int x, int y, int z) {
  const size_t lr = (size_t)ps.lr, t = (size_t)(y + 8);
  if (ps.tiled) return (((size_t)(z + 1) * plane_tiles(ps) + t / 8) * lr + (size_t)(x >> 6)) * 8 + t % 8;
  return ((size_t)(z + 1) * (size_t)(ps.ny + 1) + (size_t)(y + 1)) * lr + (size_t)(x >> 6);
}

size_t plane_cell_flags(const PlaneShape &ps, int y, int z, int *n, size_t *stride) {
  const PlaneCells c = plane_cells(ps);
  *n = kFlags;
  *stride = c.since_words;
  return (size_t)(z / (2 * kItemLayers)) * c.strips + (size_t)(y / (2 * kItemQuads));
}

}  // namespace fs3d
