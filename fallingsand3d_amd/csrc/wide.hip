// Wide multi-world tick: one launch advances a set of worlds by one tick each,
// spreading all their row quads over the whole GPU.
//
// A launch is described by a table of world entries, a prefix of their
// workgroup counts for this launch (bpre[i] = first workgroup of entry i, each
// entry padded to whole 4-wave workgroups; an entry that sits the launch out
// has none) and blk2ent, the entry of every workgroup, expanded on the device
// from the prefix.  Each workgroup reads its entry with one scalar load and its
// waves run the ordinary row-quad tick in place.  A byte grid whose final tick
// this is (k + 1 == entry.nt with entry.fin set) hashes its new state; every
// wave adds its share to hashes[entry.slot] with one atomic.  Plane grids are hashed
// at the end of the round.
//
// Used by the serving loop (continuous batching at tick granularity) and as the
// batch's third mode.  The serving loop keeps its grids as bit planes
// (wide_plane_kernel: a quarter of the bytes and no table gathers); the byte kernel
// serves batches, and requests of rows under 16 cells, whose planes would not fit
// the bytes the budget counts for them.
#include "fs3d_batch.h"
#include "plane_quad.h"
#include "tick_core.h"

namespace fs3d {
namespace {

using namespace tickcore;

// chg (optional): per hash slot, four change flags indexed by tick mod 4.  A
// launch at tick t reads the flags of ticks t-1 and t-2; when both are clear the
// world is a fixed point of both parities and the tick is not run, unless it is
// the world's final, hashed one.  Otherwise the tick runs and sets flag t when a
// cell changed.  The first workgroup of each entry clears flag t+1, which no wave
// of this launch reads or writes.  Admission sets all four flags.
template <int S>
__global__ __launch_bounds__(256) void wide_kernel(const BWorld *__restrict__ ents, const long long *__restrict__ bpre,
                                                   const int *__restrict__ blk2ent, long long blk0, int k,
                                                   const u64 *__restrict__ rule, u64 *hashes, u32 *chg) {
  const long long blk = blk0 + blockIdx.x;
  const int e = __builtin_amdgcn_readfirstlane(blk2ent[blk]);
  const BWorld w = ents[e];
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const long long wave = (blk - bpre[e]) * 4 + wid;
  const u32 t = (u32)(w.tick + (u64)k);
  const bool final_hash = k + 1 == w.nt && w.fin && hashes;
  u32 *flags = chg ? chg + (size_t)w.slot * 4 : nullptr;
  if (flags) {
    if (wave == 0 && threadIdx.x == 0) flags[(t + 1u) & 3u] = 0;
    if (!final_hash && flags[(t - 1u) & 3u] == 0 && flags[(t - 2u) & 3u] == 0) return;  // settled world
  }
  if (wave >= world_waves_dev(w.ny, w.nz, w.rqpw, (int)(t & 1u))) return;  // wave-uniform; no barriers below
  const int lane = threadIdx.x & 63;
  bool ch = false;
  if (final_hash) {
    u64 acc = tick_wave<S, true, true>(grid_of(w), grid_of(w), w.nx, w.ny, w.nz, w.lr, w.rqpw, t, wave, lane, rule, &ch);
    acc = wave_sum_u64(acc);
    if (lane == 0 && acc) atomicAdd((unsigned long long *)(hashes + w.slot), (unsigned long long)acc);
  } else {
    tick_wave<S, false, true>(grid_of(w), grid_of(w), w.nx, w.ny, w.nz, w.lr, w.rqpw, t, wave, lane, rule, &ch);
  }
  if (flags && __ballot(ch) && lane == 0) flags[t & 3u] = 1;
}

// The same tick on grids kept as bit planes, in place: lr and rqpw of an entry
// count 64-cell words.  A wave holds all rows of its row quads before it stores any.
// (Final states are hashed by wide_hash_kernel.)
//
// Serving 1500 requests of 32-256 cells a side and 10-500 ticks submitted at once:
// 187 ms with the byte kernel (336 us per launch), 31.3 ms here (44 us).  A launch over
// all of them takes up to 186 us and reads 0.44 GB; storing every word, changed or not,
// it took 222.  Several groups of row quads per wave, with the next one's rows loaded
// ahead, were slower (2: 13 %, 4: 48 %): more waves hide more than longer ones.
__global__ __launch_bounds__(256) void wide_plane_kernel(const BWorld *__restrict__ ents,
                                                         const long long *__restrict__ bpre,
                                                         const int *__restrict__ blk2ent, long long blk0, int k,
                                                         u32 *chg) {
  using namespace planedev;
  const long long blk = blk0 + blockIdx.x;
  const int e = __builtin_amdgcn_readfirstlane(blk2ent[blk]);
  const BWorld w = ents[e];
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wave = (int)(blk - bpre[e]) * 4 + wid;
  const u32 t = (u32)(w.tick + (u64)k);
  const int p = (int)(t & 1u);
  u32 *flags = chg + (size_t)w.slot * 4;
  if (wave == 0 && threadIdx.x == 0) flags[(t + 1u) & 3u] = 0;
  if (flags[(t - 1u) & 3u] == 0 && flags[(t - 2u) & 3u] == 0) return;  // settled world
  const u32 nyq = (u32)(w.ny + p + 1) >> 1, nrq = nyq * ((u32)(w.nz + p + 1) >> 1);
  const u32 q0 = (u32)wave * (u32)w.rqpw;
  if (q0 >= nrq) return;  // wave-uniform; no barriers below
  const int lane = threadIdx.x & 63;
  const int ul = lane / w.lr, seg = lane - ul * w.lr;
  const u32 q = q0 + (u32)ul, zq = q / nyq, yq = q - zq * nyq;
  const bool in = ul < w.rqpw && q < nrq;
  const int up = seg == 0 ? lane + w.lr - 1 : lane - 1, dn = seg == w.lr - 1 ? lane - (w.lr - 1) : lane + 1;
  const Planes g(w.g, (u32)w.lr * (u32)w.ny * (u32)w.nz * 16u);
  const int y0 = 2 * (int)yq - p, z0 = 2 * (int)zq - p;
  u32x4 r[4];
  u32 off[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int y = y0 + (i & 1), z = z0 + (i >> 1);
    const bool ok = in && (unsigned)y < (unsigned)w.ny && (unsigned)z < (unsigned)w.nz;
    off[i] = ok ? ((u32)(z * w.ny + y) * (u32)w.lr + (u32)seg) * 16u : kOutside;
    r[i] = g.load(off[i]);
  }
  const u32 base = variant_base(yq, zq, t);
  const int next = (in ? dn : lane) * 4;
  u32 ch;
  if (p)
    ch = quad_odd<true>(r, (u32)seg, base, (in ? up : lane) * 4, next, (w.nx & 63) == 0 && seg == 0 ? 1u : 0u);
  else
    ch = quad_even(r, (u32)seg, base);
  // in place: a word is as it was unless a block of it changed, or at odd ticks the
  // block that it shares with the word after it
  const u32 after = from_lane(next, ch) & 1u;
  const bool store = ch != 0 || (p && after);
#pragma unroll
  for (int i = 0; i < 4; i++) g.store(store, off[i], r[i]);
  if (__ballot(ch != 0) && lane == 0) flags[t & 3u] = 1;
}

// State hashes of the plane grids that finish in a round, in one launch: entry i owns
// workgroups [first[i], first[i + 1]), four lanes per word, two words of them apart.
// Hashed by the waves of their last tick, at up to 256 mixes in a row per lane, they
// made every launch in which a request finished take 28 us or more (41.5 ms for the
// 1500 requests, 37.2 with this: 24 us a round).  A workgroup adds to the entry's hash
// once: an addition to one word takes it 13 ns.
constexpr u32 kHashThreads = 1024, kHashWords = 2 * kHashThreads / 4;  // words of a workgroup
__global__ __launch_bounds__(1024) void wide_hash_kernel(const HashEntry *__restrict__ ents, int n, unsigned block0,
                                                         u64 *hashes) {
  using namespace planedev;
  const unsigned block = block0 + blockIdx.x;
  int lo = 0, hi = n;  // first of entry lo <= block < first of entry hi
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (ents[mid].first <= block) lo = mid; else hi = mid;
  }
  const HashEntry f = ents[__builtin_amdgcn_readfirstlane(lo)];
  const u32 lr = (u32)((f.nx + 63) >> 6), words = lr * (u32)f.ny * (u32)f.nz;
  const u32x4 *g = reinterpret_cast<const u32x4 *>(grid_at(f.g));
  u64 acc = 0;
#pragma unroll
  for (u32 k = 0; k < 2; k++) {
    const u32 i = (block - f.first) * kHashWords + k * (kHashThreads / 4) + (threadIdx.x >> 2);
    if (i < words) {
      const u32 row = i / lr, c = 4u * (i - row * lr) + (threadIdx.x & 3u);
      const u64 i0 = (u64)row * (u64)f.nx + (u64)(16u * c);
      acc += hash_quarter(g[i], (int)(c & 3u), min(16, f.nx - 16 * (int)c), i0, nullptr);
    }
  }
  __shared__ u64 wsum[kHashThreads / 64];
  acc = wave_sum_u64(acc);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x < 64) {
    acc = threadIdx.x < kHashThreads / 64 ? wsum[threadIdx.x] : 0;
    acc = wave_sum_u64(acc);
    if (threadIdx.x == 0 && acc) atomicAdd((unsigned long long *)(hashes + f.slot), (unsigned long long)acc);
  }
}

// Rain fills of newly admitted worlds, all in one launch: entry i owns workgroups
// [first[i], first[i + 1]), one lane per plane word.  The entry's first lane also
// clears its hash slot and sets its change flags (the first ticks of a new world
// always run).
__global__ __launch_bounds__(256) void wide_fill_kernel(const FillEntry *__restrict__ ents, int n, u64 *hashes,
                                                        u32 *chg) {
  using namespace planedev;
  int lo = 0, hi = n;  // first of entry lo <= block < first of entry hi
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (ents[mid].first <= blockIdx.x) lo = mid; else hi = mid;
  }
  const FillEntry f = ents[__builtin_amdgcn_readfirstlane(lo)];
  const u32 i = (blockIdx.x - f.first) * 256u + threadIdx.x;
  if (i == 0) {
    hashes[f.slot] = 0;
    for (int j = 0; j < 4; j++) chg[(size_t)f.slot * 4 + j] = 1u;
  }
  const u32 lr = (u32)((f.nx + 63) >> 6);
  if (i >= lr * (u32)f.ny * (u32)f.nz) return;
  const u32 row = i / lr, seg = i - row * lr, z = row / (u32)f.ny;
  const int m = min(64, f.nx - 64 * (int)seg);
  u32x4 v = u32x4{0u, 0u, 0u, 0u};  // z = 0: the floor
  if (z > 0) {
    const bool rain = z >= (u32)max(1, f.nz >> 1);
    const u64 i0 = (u64)row * (u64)f.nx + (u64)(64u * seg);
    for (int j = 0; j < 32; j++) {
      const u32 bit = 1u << pair_bit(j);
      const int x = 2 * j;
      if (x < m) {
        v.x |= bit;
        if (rain && dmix64(f.seed + (i0 + (u64)x + 1) * kGamma) < f.thr) v.z |= bit;
      }
      if (x + 1 < m) {
        v.y |= bit;
        if (rain && dmix64(f.seed + (i0 + (u64)x + 2) * kGamma) < f.thr) v.w |= bit;
      }
    }
  }
  reinterpret_cast<u32x4 *>(f.g)[i] = v;
}

// out[i] = hashes[slots[i]] (out: pinned host memory).
__global__ void gather_hashes_kernel(const u64 *__restrict__ hashes, const int *__restrict__ slots, int n, u64 *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = hashes[slots[i]];
}

// blk2ent[b] = i for every workgroup b of entry i.
__global__ __launch_bounds__(256) void expand_kernel(const long long *__restrict__ bpre, int n, int *blk2ent) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    for (long long b = bpre[i]; b < bpre[i + 1]; b++) blk2ent[b] = i;
}

// The workgroup -> entry tables of K launches at once: launch k's workgroups are
// [koff[k], koff[k+1]) of blk2ent and its prefix is bpre[k*(n+1) .. k*(n+1)+n];
// one thread per workgroup finds its entry by binary search (the last i with
// bpre[i] <= b: an entry with blocks covering b has bpre[i+1] > b).
__global__ __launch_bounds__(256) void expand_round_kernel(const long long *__restrict__ bpre, int n, int K,
                                                           const long long *__restrict__ koff, long long total,
                                                           int *blk2ent) {
  for (long long gb = (long long)blockIdx.x * blockDim.x + threadIdx.x; gb < total;
       gb += (long long)gridDim.x * blockDim.x) {
    int k = 0;
    while (k + 1 < K && koff[k + 1] <= gb) k++;
    const long long b = gb - koff[k];
    const long long *pre = bpre + (size_t)k * (n + 1);
    int lo = 0, hi = n;  // pre[lo] <= b < pre[hi]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (pre[mid] <= b) lo = mid; else hi = mid;
    }
    blk2ent[gb] = lo;
  }
}

// hashes[ents[i].slot] = 0 for i < n (before a final tick accumulates into them).
__global__ void zero_slots_kernel(u64 *hashes, const BWorld *__restrict__ ents, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) hashes[ents[i].slot] = 0;
}

}  // namespace

hipError_t launch_wide(int seg, const BWorld *ents, const long long *bpre, const int *blk2ent, long long blk0,
                       long long blocks, int k, const u64 *rule, u64 *hashes, hipStream_t s, u32 *chg) {
  if (blocks <= 0) return hipSuccess;
  const dim3 grid((unsigned)blocks);
  switch (seg) {
    case 8:
      hipLaunchKernelGGL(wide_kernel<8>, grid, dim3(256), 0, s, ents, bpre, blk2ent, blk0, k, rule, hashes, chg);
      break;
    case 16:
      hipLaunchKernelGGL(wide_kernel<16>, grid, dim3(256), 0, s, ents, bpre, blk2ent, blk0, k, rule, hashes, chg);
      break;
    default:
      hipLaunchKernelGGL(wide_kernel<32>, grid, dim3(256), 0, s, ents, bpre, blk2ent, blk0, k, rule, hashes, chg);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_wide_planes(const BWorld *ents, const long long *bpre, const int *blk2ent, long long blk0,
                              long long blocks, int k, hipStream_t s, u32 *chg) {
  if (blocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(wide_plane_kernel, dim3((unsigned)blocks), dim3(256), 0, s, ents, bpre, blk2ent, blk0, k, chg);
  return hipGetLastError();
}

unsigned hash_blocks(size_t words) { return (unsigned)((words + kHashWords - 1) / kHashWords); }

hipError_t launch_wide_hash(const HashEntry *ents, int n, unsigned blocks, u64 *hashes, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  constexpr unsigned kMax = (1u << 22) - 1u;  // a launch takes fewer than 2^32 threads
  for (unsigned b = 0; b < blocks; b += kMax) {
    hipLaunchKernelGGL(wide_hash_kernel, dim3(blocks - b < kMax ? blocks - b : kMax), dim3(kHashThreads), 0, s, ents, n,
                       b, hashes);
    if (const hipError_t e = hipGetLastError()) return e;
  }
  return hipSuccess;
}

hipError_t launch_wide_fill(const FillEntry *ents, int n, unsigned blocks, u64 *hashes, u32 *chg, hipStream_t s) {
  hipLaunchKernelGGL(wide_fill_kernel, dim3(blocks), dim3(256), 0, s, ents, n, hashes, chg);
  return hipGetLastError();
}

hipError_t launch_gather_hashes(const u64 *hashes, const int *slots, int n, u64 *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(gather_hashes_kernel, dim3((n + 255) / 256), dim3(256), 0, s, hashes, slots, n, out);
  return hipGetLastError();
}

hipError_t launch_expand(const long long *bpre, int n, int *blk2ent, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int grid = (n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024;
  hipLaunchKernelGGL(expand_kernel, dim3(grid), dim3(256), 0, s, bpre, n, blk2ent);
  return hipGetLastError();
}

hipError_t launch_expand_round(const long long *bpre, int n, int K, const long long *koff, long long total,
                               int *blk2ent, hipStream_t s) {
  if (total <= 0 || n <= 0) return hipSuccess;
  const long long want = (total + 255) / 256;
  const unsigned grid = (unsigned)(want < 4096 ? want : 4096);
  hipLaunchKernelGGL(expand_round_kernel, dim3(grid), dim3(256), 0, s, bpre, n, K, koff, total, blk2ent);
  return hipGetLastError();
}

hipError_t launch_zero_slots(u64 *hashes, const BWorld *ents, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(zero_slots_kernel, dim3((n + 255) / 256), dim3(256), 0, s, hashes, ents, n);
  return hipGetLastError();
}

long long world_waves(const BWorld &w, int p) { return world_waves_dev(w.ny, w.nz, w.rqpw, p); }

long long world_blocks(const BWorld &w, int p) { return (world_waves(w, p) + 3) / 4; }

}  // namespace fs3d
