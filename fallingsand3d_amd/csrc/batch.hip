// Batched worlds: many independent grids of uneven sizes stepped by one
// persistent kernel on bit planes.
//
// A workgroup takes the next world from an atomic queue (largest first), packs
// its grid into bit planes (plane_core.h), runs all requested ticks there and
// writes the cells back: in LDS when the world's planes fit the workgroup's share,
// else in a plane scratch of its own in device memory.  The waves sweep the
// world's row quads in place (a quad's four rows are loaded whole before any is
// stored, and a tick's quads are disjoint) with a workgroup barrier between
// ticks.  Worlds whose planes fit a wave's share of the LDS are taken by single
// waves afterwards, without barriers.
//
// Why: the ticks of a world this small never leave the CU, so the kernel is bound
// by the rule's instructions (about 350 per 2048 blocks) and by waves idle at the
// barriers of worlds with few row quads.  On bytes it was bound by the table
// gathers and by cache traffic of in-place byte grids: 4096 worlds of 16-128 cells
// a side (0.61 G voxels), fill and 500 ticks: 26.6-28.7 -> 5.4 ms.  Workgroup sizes
// on that batch, 10 ticks: 1.64 / 1.08 / 1.16 ms at 256 / 512 / 1024 threads.
//
// The reference has nothing of the kind (one world, one process, no simulation);
// this is the batching mode the tick is required to support.
#include <algorithm>

#include "fs3d_batch.h"
#include "plane_quad.h"

namespace fs3d {
namespace {

using namespace planedev;

// A world's planes in LDS: words behind a zero word, which rows outside the grid
// read (STATIC); their stores are dropped.
struct LdsPlanes {
  u32x4 *w;
  __device__ __forceinline__ u32x4 load(u32 i, bool ok) const { return w[ok ? i + 1u : 0u]; }
  __device__ __forceinline__ void store(u32 i, bool ok, u32x4 v) const {
    if (ok) w[i + 1u] = v;
  }
};

// The same in device memory.
struct GlobalPlanes {
  Planes p;
  __device__ __forceinline__ u32x4 load(u32 i, bool ok) const { return p.load(ok ? i * 16u : kOutside); }
  __device__ __forceinline__ void store(u32 i, bool ok, u32x4 v) const { p.store(ok ? i * 16u : kOutside, v); }
};

// The queue hands a wave one world, so its table entry is the same in every lane:
// told so, the compiler keeps it, and a buffer made from it, in scalar registers.
__device__ __forceinline__ u64 uniform64(u64 v) {
  return ((u64)(u32)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
         (u32)__builtin_amdgcn_readfirstlane((int)(u32)v);
}
__device__ __forceinline__ BWorld world_at(const BWorld *worlds, int wi) {
  BWorld w = worlds[wi];
  w.g = (u8 *)(uintptr_t)uniform64((u64)(uintptr_t)w.g);
  w.nx = __builtin_amdgcn_readfirstlane(w.nx);
  w.ny = __builtin_amdgcn_readfirstlane(w.ny);
  w.nz = __builtin_amdgcn_readfirstlane(w.nz);
  w.tick = uniform64(w.tick);
  w.poff = uniform64(w.poff);
  return w;
}

// Orders a wave's accesses for its own lanes, which pass planes to each other through LDS
// from packing to the ticks and to unpacking: no instruction, since the LDS answers a wave
// in order, but the compiler keeps to it.
__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

struct Geo {
  int nx, ny, nz, lr, upw;
  int ul, seg, prev, next;  // the lane's row quad of a group, word, ring neighbours
  bool in;
  u32 wall;
};

__device__ __forceinline__ Geo geo_of(const BWorld &w, int lane) {
  Geo g;
  g.nx = w.nx, g.ny = w.ny, g.nz = w.nz;
  g.lr = (w.nx + 63) >> 6;
  g.upw = 64 / g.lr;
  g.ul = lane / g.lr;
  g.seg = lane - g.ul * g.lr;
  g.in = g.ul < g.upw;
  const int up = g.seg == 0 ? lane + g.lr - 1 : lane - 1, dn = g.seg == g.lr - 1 ? lane - (g.lr - 1) : lane + 1;
  g.prev = (g.in ? up : lane) * 4;
  g.next = (g.in ? dn : lane) * 4;
  g.wall = (w.nx & 63) == 0 && g.seg == 0 ? 1u : 0u;
  return g;
}

// One tick of parity P: row-quad groups first, first + stride, ...  True when a
// block of this lane changed.
template <int P, class Mem>
__device__ __forceinline__ bool batch_tick(const Mem &mem, const Geo &g, u32 t, int first, int stride) {
  const u32 nyq = (u32)(g.ny + P + 1) >> 1, nrq = nyq * ((u32)(g.nz + P + 1) >> 1);
  u32 chg = 0;
  for (u32 q0 = (u32)first * (u32)g.upw; q0 < nrq; q0 += (u32)stride * (u32)g.upw) {
    const u32 q = q0 + (u32)g.ul;
    const bool in = g.in && q < nrq;
    const u32 zq = q / nyq, yq = q - zq * nyq;
    const int y0 = 2 * (int)yq - P, z0 = 2 * (int)zq - P;
    u32x4 r[4];
    u32 idx[4];
    bool ok[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int y = y0 + (i & 1), z = z0 + (i >> 1);
      ok[i] = in && (P == 0 || ((i & 1) || y >= 0)) && (P == 0 || ((i >> 1) || z >= 0)) && y < g.ny && z < g.nz;
      idx[i] = (u32)(z * g.ny + y) * (u32)g.lr + (u32)g.seg;
      r[i] = mem.load(idx[i], ok[i]);
    }
    const u32 base = variant_base(yq, zq, t);
    if constexpr (P)
      chg |= quad_odd<true>(r, (u32)g.seg, base, g.prev, g.next, g.wall);
    else
      chg |= quad_even(r, (u32)g.seg, base);
#pragma unroll
    for (int i = 0; i < 4; i++) mem.store(idx[i], ok[i], r[i]);
  }
  return chg != 0;
}

// Bytes to planes and back by `lanes` lanes, of which this is `id`; unpacking
// returns the lane's share of the state hash when hash is set.
template <class Mem>
__device__ __forceinline__ bool batch_pack(const Mem &mem, const u8 *bytes, const Geo &g, u32 words, u32 id,
                                           u32 lanes) {
  bool res = false;
  for (u32 i0 = 0; i0 < words; i0 += lanes) {
    const u32 i = i0 + id;
    const bool ok = i < words;
    const u32 row = (ok ? i : 0u) / (u32)g.lr, c = (ok ? i : 0u) - row * (u32)g.lr;
    const u32x4 v = word_from_bytes(bytes + (size_t)row * (u32)g.nx + 64u * c, min(64, g.nx - 64 * (int)c), &res);
    mem.store(i, ok, v);
  }
  return res;
}

template <class Mem>
__device__ __forceinline__ u64 batch_unpack(const Mem &mem, u8 *bytes, const Geo &g, u32 words, u32 id, u32 lanes,
                                            bool keep, bool hash) {
  u64 acc = 0;
  for (u32 i = id; i < 4u * words; i += lanes) {
    const u32 qpr = 4u * (u32)g.lr, row = i / qpr, c = i - row * qpr;
    const int m = min(16, g.nx - 16 * (int)c);
    if (m <= 0) continue;
    const size_t i0 = (size_t)row * (u32)g.nx + 16u * c;
    const u32x4 v = mem.load(i >> 2, true);
    if (hash) acc += hash_quarter(v, (int)(c & 3u), m, i0, keep ? bytes + i0 : nullptr);
    u32 d[4];
    unpack_quarter(v, (int)(c & 3u), d);
    store_quarter(bytes + i0, m, d, keep);
  }
  return acc;
}

// A world's ticks by a whole workgroup.
template <int NT, class Mem>
__device__ __forceinline__ void run_world(const Mem &mem, const BWorld &w, u32 words, int nticks, bool settle,
                                          u64 *hash_out, u64 *s_sum) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const Geo g = geo_of(w, lane);
  u8 *const bytes = grid_of(w);
  const bool keep = __syncthreads_or(batch_pack(mem, bytes, g, words, threadIdx.x, NT));
  int quiet = 0;  // consecutive ticks in which no cell of the world changed
  for (int k = 0; k < nticks; k++) {
    // Two quiet ticks in a row (one of each parity) make the state a fixed point
    // of both parities, whatever the variants.
    if (settle && quiet >= 2) break;
    const u32 t = (u32)(w.tick + (u64)k);
    const bool ch = (t & 1u) ? batch_tick<1>(mem, g, t, wid, NW) : batch_tick<0>(mem, g, t, wid, NW);
    quiet = __syncthreads_or(ch) ? 0 : quiet + 1;
  }
  u64 acc = batch_unpack(mem, bytes, g, words, threadIdx.x, NT, keep, hash_out != nullptr);
  if (hash_out) {
    acc = wave_sum_u64(acc);
    if (lane == 0) s_sum[wid] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      u64 tot = 0;
#pragma unroll
      for (int i = 0; i < NW; i++) tot += s_sum[i];
      *hash_out = tot;
    }
  }
  __syncthreads();
}

// order: world indices by plane words, largest first; the first n_wide of them
// are taken by workgroups, the others by waves.  planes: plane scratch of the
// worlds over lds_words.
template <int NT>
__global__ __launch_bounds__(NT, 4) void batch_kernel(BWorld *worlds, const int *order, int n_wide, int n, int nticks,
                                                      u32 *queue, u32x4 *planes, u32 lds_words,
                                                      u64 *hashes, int flags) {
  constexpr int NW = NT / 64;
  extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
  __shared__ int s_idx;
  __shared__ u64 s_sum[NW];
  const bool want_hash = flags & kBatchHash, settle = flags & kBatchSettle;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (;;) {
    if (threadIdx.x == 0) {
      s_idx = (int)atomicAdd(queue, 1u);
      lds[0] = u32x4{0u, 0u, 0u, 0u};
    }
    __syncthreads();
    // The queue index is the same for the whole workgroup; readfirstlane makes
    // that visible to the compiler, so the loop exit below is a uniform (scalar)
    // branch and every wave meets the same barriers.
    const int idx = __builtin_amdgcn_readfirstlane(s_idx);
    __syncthreads();
    if (idx >= n_wide) break;
    const int wi = __builtin_amdgcn_readfirstlane(order[idx]);
    const BWorld w = world_at(worlds, wi);
    const u32 words = (u32)((w.nx + 63) >> 6) * (u32)w.ny * (u32)w.nz;
    u64 *const out = want_hash ? hashes + wi : nullptr;
    if (words <= lds_words)
      run_world<NT>(LdsPlanes{lds}, w, words, nticks, settle, out, s_sum);
    else
      run_world<NT>(GlobalPlanes{Planes(planes + w.poff, words * 16u)}, w, words, nticks, settle, out, s_sum);
    if (threadIdx.x == 0) worlds[wi].tick = w.tick + (u64)nticks;
    // Rejoins thread 0 before the loop's own thread-0 block: without a convergent
    // operation between the two, the compiler threads the one into the other and
    // the other lanes run the barriers above without it.
    __syncthreads();
  }
  // ---- small worlds, one per wave ----
  const LdsPlanes mem{lds + (size_t)wid * batch_wave_words(lds_words, NW)};
  if (lane == 0) mem.w[0] = u32x4{0u, 0u, 0u, 0u};
  for (;;) {
    u32 got = 0;
    if (lane == 0) got = atomicAdd(queue + 1, 1u);
    const int idx = n_wide + (int)__builtin_amdgcn_readfirstlane((int)got);
    if (idx >= n) break;
    const int wi = __builtin_amdgcn_readfirstlane(order[idx]);
    const BWorld w = world_at(worlds, wi);
    const u32 words = (u32)((w.nx + 63) >> 6) * (u32)w.ny * (u32)w.nz;
    const Geo g = geo_of(w, lane);
    u8 *const bytes = grid_of(w);
    const bool keep = __any(batch_pack(mem, bytes, g, words, lane, 64));
    wave_fence();
    int quiet = 0;
    for (int k = 0; k < nticks; k++) {
      if (settle && quiet >= 2) break;
      const u32 t = (u32)(w.tick + (u64)k);
      const bool ch = (t & 1u) ? batch_tick<1>(mem, g, t, 0, 1) : batch_tick<0>(mem, g, t, 0, 1);
      wave_fence();
      quiet = __any(ch) ? 0 : quiet + 1;
    }
    const u64 acc = wave_sum_u64(batch_unpack(mem, bytes, g, words, lane, 64, keep, want_hash));
    if (lane == 0) {
      if (want_hash) hashes[wi] = acc;
      worlds[wi].tick = w.tick + (u64)nticks;
    }
    __builtin_amdgcn_wave_barrier();  // rejoins lane 0, as above
  }
}

// One workgroup per world: hash of the current grid.
__global__ __launch_bounds__(256) void batch_hash_kernel(const BWorld *worlds, int n, u64 *hashes) {
  __shared__ u64 s_sum[4];
  for (int wi = blockIdx.x; wi < n; wi += gridDim.x) {
    const BWorld w = worlds[wi];
    const size_t cnt = (size_t)w.nx * w.ny * w.nz;
    u64 acc = 0;
    for (size_t i = threadIdx.x; i < cnt; i += 256) {
      const u32 v = grid_of(w)[i];
      if (v) acc += dmix64(((u64)i << 8) | v);
    }
    acc = wave_sum_u64(acc);
    if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) hashes[wi] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
    __syncthreads();
  }
}

// Rain fill of every world (same cell rule as the single-world fill).
__global__ __launch_bounds__(256) void batch_fill_rain_kernel(const BWorld *worlds, int n, const u64 *seeds,
                                                              const u64 *thr) {
  for (int wi = blockIdx.y; wi < n; wi += gridDim.y) {
    const BWorld w = worlds[wi];
    const u64 layer = (u64)w.nx * w.ny, cnt = layer * w.nz, rain = (u64)max(1, w.nz >> 1) * layer;
    const u64 seed = seeds[wi], th = thr[wi];
    for (u64 i = 16 * ((u64)blockIdx.x * 256 + threadIdx.x); i < cnt; i += 16 * 256 * (u64)gridDim.x)
      tickcore::fill_rain16(grid_of(w), i, cnt, layer, rain, seed, th);
  }
}

__global__ void reset_u32_kernel(u32 *p) {
  if (threadIdx.x < 2) p[threadIdx.x] = 0u;
}

// Dynamic LDS of a workgroup: its share of the CU at 1024 threads per CU.
size_t lds_bytes(int threads) { return (size_t)(158 * 1024) * (size_t)threads / 1024; }

}  // namespace

bool batch_config_ok(int seg, int threads, int groups) {
  const bool t_ok = threads == 256 || threads == 512 || threads == 1024;
  const bool g_ok = groups == 1 || groups == 2 || groups == 4;
  if (seg == 8 || seg == 16) return t_ok && g_ok;
  return seg == 32 && threads == 256 && groups == 1;
}

u32 batch_lds_words(int threads) { return (u32)(lds_bytes(threads) / 16) - 1u; }

int batch_occupancy(int threads) { return 1024 / threads; }

hipError_t launch_batch(int threads, BWorld *worlds, const int *order, int n_wide, int n, int nticks, u32 *queue,
                        void *planes, u64 *hashes, int flags, int grid, hipStream_t s) {
  hipLaunchKernelGGL(reset_u32_kernel, dim3(1), dim3(64), 0, s, queue);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  u32x4 *const pl = static_cast<u32x4 *>(planes);
  const size_t lds = lds_bytes(threads);
  const u32 lw = batch_lds_words(threads);
  switch (threads) {
    case 256:
      hipLaunchKernelGGL(batch_kernel<256>, dim3(grid), dim3(256), lds, s, worlds, order, n_wide, n, nticks, queue, pl,
                         lw, hashes, flags);
      break;
    case 512:
      hipLaunchKernelGGL(batch_kernel<512>, dim3(grid), dim3(512), lds, s, worlds, order, n_wide, n, nticks, queue, pl,
                         lw, hashes, flags);
      break;
    default:
      hipLaunchKernelGGL(batch_kernel<1024>, dim3(grid), dim3(1024), lds, s, worlds, order, n_wide, n, nticks, queue,
                         pl, lw, hashes, flags);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_batch_hash(const BWorld *worlds, int n, u64 *hashes, hipStream_t s) {
  const int grid = n < 8192 ? n : 8192;
  hipLaunchKernelGGL(batch_hash_kernel, dim3(grid > 0 ? grid : 1), dim3(256), 0, s, worlds, n, hashes);
  return hipGetLastError();
}

hipError_t launch_batch_fill_rain(const BWorld *worlds, int n, const u64 *seeds, const u64 *thr, size_t max_cells,
                                  hipStream_t s) {
  unsigned gx = (unsigned)std::min<size_t>((max_cells + 4095) / 4096, 64);
  unsigned gy = (unsigned)std::min(n, 65535);
  hipLaunchKernelGGL(batch_fill_rain_kernel, dim3(gx ? gx : 1, gy ? gy : 1), dim3(256), 0, s, worlds, n, seeds, thr);
  return hipGetLastError();
}

}  // namespace fs3d
