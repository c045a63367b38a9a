// Bit-plane kernels: packing, unpacking, single ticks, pairs of ticks and the
// state hash on two bits per cell (plane_core.h has the layout and the rule).
//
// A plane grid is rows of lr = ceil(nx / 64) words of 16 bytes, v[z][y][word].
// One lane holds one word of each of a row quad's four rows.
//
// What this replaces: the byte kernels move 2 bytes per voxel-update and gather
// one 8-byte table entry per block (510 vector instructions per 1024 blocks and
// the gathers' latency).  Here a single tick moves 0.5 bytes and takes about 335
// instructions per 2048 blocks, none of them a load, and a pair of ticks moves
// about 0.3 bytes per voxel-update.  Dense ticks on an MI355X, us per tick, byte
// kernels / single plane ticks / plane pairs:
//   512^3            42 / 12.2 / 9.3      (10.99 and 14.5 T voxel-updates/s)
//   1000 x 701 x 603 186 (fused pairs 182) / 34 / 22.4
//   2048^3           3070 (fused pairs 2300) / 770 / 416
// Single ticks are bound by memory (2048^3: 4.3 GB in 770 us, 5.6 TB/s), pairs by
// their instructions (1.3 evaluations per row quad and tick with the halo).
#include "plane_quad.h"

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

// ---- single tick ----------------------------------------------------------------
template <bool WALL>
__global__ __launch_bounds__(256) void plane_tick_kernel(PlaneArgs a) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const u64 t64 = tick_of(a);
  const u32 t = (u32)t64;
  const int p = (int)(t & 1u);
  const int nyq = (a.ny + p + 1) >> 1, nzq = (a.nz + p + 1) >> 1;
  const int first = ((int)blockIdx.x * 4 + wv) * a.upw;
  const int zq = (int)blockIdx.z * 65535 + (int)blockIdx.y;
  if (__builtin_amdgcn_readfirstlane(first) >= nyq || zq >= nzq) return;
  const Lane L = lane_of(a, first, lane);
  const Planes src(a.src, a.bytes), dst(a.dst, a.bytes);
  const int y0 = 2 * L.unit - p, z0 = 2 * zq - p;
  u32x4 r[4];
  u32 off[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int y = y0 + (i & 1), z = z0 + (i >> 1);
    const bool ok = L.in && (unsigned)y < (unsigned)a.ny && (unsigned)z < (unsigned)a.nz;
    off[i] = ok ? ((u32)(z * a.ny + y) * (u32)a.lr + (u32)L.seg) * 16u : kOutside;
    r[i] = src.load(off[i]);
  }
  const u32 base = variant_base((u32)L.unit, (u32)zq, t);
  if (p)
    quad_odd<WALL>(r, (u32)L.seg, base, L.prev, L.next, L.wall);
  else
    quad_even(r, (u32)L.seg, base);
#pragma unroll
  for (int i = 0; i < 4; i++) dst.store(off[i], r[i]);
}

// ---- a pair of ticks --------------------------------------------------------------
// Ticks t (odd) and t + 1 in one pass.  A lane owns K even-parity row quads along
// y (a strip, 2K rows) and sweeps z row-quads [Z0, Z1).  Odd row quad i of layer
// pair s covers rows 2 (Y0 + i) - 1 and + 0 and layers 2s - 1 and 2s, so the even
// row quad (Y0 + j, b) takes its four rows from odd quads j and j + 1 of s = b
// (their upper layers) and s = b + 1 (their lower ones).  Everything stays in
// registers: the upper layers of the previous s (top), and the quad before.
template <bool WALL, int K>
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
  const Lane L = lane_of(a, yt * a.upw, lane);
  const int Y0 = L.unit * K;
  const u32 seg = (u32)L.seg;
  const Planes src(a.src, a.bytes), dst(a.dst, a.bytes);
  const u32 row_bytes = (u32)a.lr * 16u, layer_bytes = row_bytes * (u32)a.ny;
  const u32 lane_off = (u32)(2 * Y0) * row_bytes + seg * 16u;  // row 2 Y0 of a layer
  auto offset = [&](int dy, int z) {
    const bool ok = L.in && (unsigned)(2 * Y0 + dy) < (unsigned)a.ny && (unsigned)z < (unsigned)a.nz;
    return ok ? lane_off + (u32)dy * row_bytes + (u32)z * layer_bytes : kOutside;
  };
  u32x4 top[2 * K];
  u32x4 nx[4];
#pragma unroll
  for (int r = 0; r < 4; r++) nx[r] = src.load(offset(-1 + (r & 1), 2 * Z0 - 1 + (r >> 1)));
  for (int s = Z0; s <= Z1; s++) {
    u32x4 lowp, upp;  // upper row of the odd quad before: its lower and upper layer
#pragma unroll
    for (int i = 0; i <= K; i++) {
      u32x4 q[4];
#pragma unroll
      for (int r = 0; r < 4; r++) q[r] = nx[r];
      const int in = i < K ? i + 1 : 0, sn = i < K ? s : s + 1;
#pragma unroll
      for (int r = 0; r < 4; r++) nx[r] = src.load(offset(2 * in - 1 + (r & 1), 2 * sn - 1 + (r >> 1)));
      // One quad at a time: left alone, the scheduler interleaves the evaluations
      // of several, for which there are no registers.
      __builtin_amdgcn_sched_barrier(0);
      quad_odd<WALL>(q, seg, variant_base((u32)(Y0 + i), (u32)s, t), L.prev, L.next, L.wall);
      __builtin_amdgcn_sched_barrier(0);
      if (i > 0) {
        if (s > Z0) {
          u32x4 e[4] = {top[2 * i - 2], top[2 * i - 1], lowp, q[0]};
          quad_even(e, seg, variant_base((u32)(Y0 + i - 1), (u32)(s - 1), t + 1u));
#pragma unroll
          for (int r = 0; r < 4; r++) dst.store(offset(2 * i - 2 + (r & 1), 2 * (s - 1) + (r >> 1)), e[r]);
        }
        top[2 * i - 2] = upp;
        top[2 * i - 1] = q[2];
      }
      lowp = q[1];
      upp = q[3];
    }
  }
}

// ---- bytes <-> planes --------------------------------------------------------------
// One lane per word: 64 bytes of a row.  *reserved is set when a byte >= 4 is seen
// (the planes hold STATIC for it).
__global__ __launch_bounds__(256) void plane_pack_kernel(const u8 *g, u32x4 *out, int nx, int lr, size_t words,
                                                         u32 *reserved) {
  bool any = false;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < words; i += (size_t)gridDim.x * 256) {
    const size_t row = i / (u32)lr;
    const int x0 = (int)(i - row * (u32)lr) * 64, m = min(64, nx - x0);
    // loads may run up to 63 bytes past the last row, into the guard bytes
    out[i] = word_from_bytes(g + row * (size_t)nx + x0, m, &any);
  }
  if (__any(any) && (threadIdx.x & 63) == 0) *reserved = 1u;
}

// Planes to bytes, four lanes per word so that a wave stores 1 KiB in a row.
__global__ __launch_bounds__(256) void plane_unpack_kernel(const u32x4 *in, u8 *g, int nx, int lr, size_t quarters,
                                                           const u32 *reserved) {
  const bool keep = *reserved != 0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < quarters; i += (size_t)gridDim.x * 256) {
    const u32 qpr = 4u * (u32)lr;
    const size_t row = i / qpr;
    const int c = (int)(i - row * qpr), m = min(16, nx - 16 * c);
    if (m <= 0) continue;
    u8 *p = g + row * (size_t)nx + 16 * c;
    u32 d[4];
    unpack_quarter(in[i >> 2], c & 3, d);
    store_quarter(p, m, d, keep);  // reserved cells hold their bytes (they never move)
  }
}

// State hash of a plane grid, four lanes per word: each lane mixes its quarter's
// non-empty cells.  With *reserved, STATIC cells are read from the bytes.
__global__ __launch_bounds__(256) void plane_hash_kernel(const u32x4 *in, const u8 *g, int nx, int lr, size_t quarters,
                                                         const u32 *reserved, u64 *parts) {
  const bool bytes = *reserved != 0;
  u64 acc = 0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < quarters; i += (size_t)gridDim.x * 256) {
    const u32 qpr = 4u * (u32)lr;
    const size_t row = i / qpr;
    const int c = (int)(i - row * qpr), m = min(16, nx - 16 * c);
    const u64 i0 = row * (u64)nx + (u64)(16 * c);
    acc += hash_quarter(in[i >> 2], c & 3, m, i0, bytes ? g + i0 : nullptr);
  }
  __shared__ u64 wsum[4];
  acc = wave_sum_u64(acc);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const u64 tot = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    if (tot) atomicAdd((unsigned long long *)(parts + (size_t)(blockIdx.x % kHashParts) * kHashStride),
                       (unsigned long long)tot);
  }
}

// One cell set by the host.
__global__ void plane_set_kernel(u32 *planes, size_t word, int x, u32 v, u32 *reserved) {
  if (threadIdx.x != 0) return;
  if (v >= 4u) *reserved = 1u;
  const u32 code = (v >= 4u ? (u32)FS3D_STATIC : v) ^ 1u;
  u32 *w = planes + 4 * word + (x & 1);
  const u32 m = 1u << pair_bit((x & 63) >> 1);
  w[0] = (code & 1u) ? w[0] | m : w[0] & ~m;
  w[2] = (code & 2u) ? w[2] | m : w[2] & ~m;
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

hipError_t launch_plane_tick(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             hipStream_t s) {
  PlaneArgs a{};
  fill_args(a, ps);
  a.src = static_cast<const u32x4 *>(src);
  a.dst = static_cast<u32x4 *>(dst);
  a.t = t;
  a.tick_dev = tick_dev;
  a.k_off = k_off;
  const int nyq = (ps.ny + 2) >> 1, nzq = (ps.nz + 2) >> 1, per = 4 * a.upw;
  const dim3 grid((unsigned)((nyq + per - 1) / per), (unsigned)std::min(nzq, 65535), (unsigned)((nzq + 65534) / 65535));
  if (ps.nx % 64 == 0)
    hipLaunchKernelGGL(plane_tick_kernel<true>, grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(plane_tick_kernel<false>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_plane_pair(const PlaneShape &ps, const void *src, void *dst, u64 t, const u64 *tick_dev, u32 k_off,
                             int k, int zlen, hipStream_t s) {
  PlaneArgs a{};
  fill_args(a, ps);
  a.src = static_cast<const u32x4 *>(src);
  a.dst = static_cast<u32x4 *>(dst);
  a.t = t;
  a.tick_dev = tick_dev;
  a.k_off = k_off;
  a.zlen = zlen;
  const int nyq = (ps.ny + 1) >> 1, nzq = (ps.nz + 1) >> 1;
  const int strips = (nyq + k - 1) / k;
  a.ytiles = (strips + a.upw - 1) / a.upw;
  const long long waves = (long long)a.ytiles * ((nzq + zlen - 1) / zlen);
  const dim3 grid((unsigned)((waves + 3) / 4));
  const bool wall = ps.nx % 64 == 0;
  switch (k) {
    case 1:
      if (wall) hipLaunchKernelGGL((plane_pair_kernel<true, 1>), grid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((plane_pair_kernel<false, 1>), grid, dim3(256), 0, s, a);
      break;
    case 2:
      if (wall) hipLaunchKernelGGL((plane_pair_kernel<true, 2>), grid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((plane_pair_kernel<false, 2>), grid, dim3(256), 0, s, a);
      break;
    default:
      if (wall) hipLaunchKernelGGL((plane_pair_kernel<true, 4>), grid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((plane_pair_kernel<false, 4>), grid, dim3(256), 0, s, a);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_plane_pack(const PlaneShape &ps, const u8 *g, void *planes, u32 *reserved, hipStream_t s) {
  const size_t words = plane_words(ps);
  const unsigned grid = (unsigned)std::min<size_t>((words + 255) / 256, 1u << 20);
  hipLaunchKernelGGL(plane_pack_kernel, dim3(grid), dim3(256), 0, s, g, static_cast<u32x4 *>(planes), ps.nx, ps.lr,
                     words, reserved);
  return hipGetLastError();
}

hipError_t launch_plane_unpack(const PlaneShape &ps, const void *planes, u8 *g, const u32 *reserved, hipStream_t s) {
  const size_t quarters = 4 * plane_words(ps);
  const unsigned grid = (unsigned)std::min<size_t>((quarters + 255) / 256, 1u << 20);
  hipLaunchKernelGGL(plane_unpack_kernel, dim3(grid), dim3(256), 0, s, static_cast<const u32x4 *>(planes), g, ps.nx,
                     ps.lr, quarters, reserved);
  return hipGetLastError();
}

hipError_t launch_plane_hash(const PlaneShape &ps, const void *planes, const u8 *g, const u32 *reserved, u64 *parts,
                             hipStream_t s) {
  const size_t quarters = 4 * plane_words(ps);
  const unsigned grid = (unsigned)std::min<size_t>((quarters + 255) / 256, 8192);
  hipLaunchKernelGGL(plane_hash_kernel, dim3(grid), dim3(256), 0, s, static_cast<const u32x4 *>(planes), g, ps.nx,
                     ps.lr, quarters, reserved, parts);
  return hipGetLastError();
}

hipError_t launch_plane_set(const PlaneShape &ps, void *planes, int x, int y, int z, u8 v, u32 *reserved,
                            hipStream_t s) {
  const size_t word = ((size_t)z * ps.ny + y) * ps.lr + (size_t)(x >> 6);
  hipLaunchKernelGGL(plane_set_kernel, dim3(1), dim3(64), 0, s, static_cast<u32 *>(planes), word, x, (u32)v, reserved);
  return hipGetLastError();
}

}  // namespace fs3d
