// Single cells set and read by the host, and results handed to it.
//
// An editor's calls are one cell or one hash each, and what they take is latency.
// Each is one launch, and what it returns, and that it is done, the kernel writes to
// pinned memory, where the host looks for it.  Three cells set, a tick, a cell read
// and a hashed tick of 48 x 37 x 29 take 61 us; copying bytes, marking masks in a
// launch of its own and waiting for the stream each time they took 98.
#include "plane_quad.h"

namespace fs3d {
namespace {

using planedev::pair_bit;

// One lane: the byte, the change bits of the segments around it at both parities
// (edge words at edge_off), and where the planes hold the state, the cell's bits and
// its item's change flags.
__global__ void set_cell_kernel(CellEdit e, Note n) {
  if (threadIdx.x != 0) return;
  *e.cell = (u8)e.value;
#pragma unroll
  for (int p = 0; p < 2; p++) {
    e.masks[p][e.idx[p]] |= e.bits;
    e.masks[p][e.edge_off + e.idx[p]] |= e.bits | (e.bits << 1);
  }
  if (e.planes) {
    for (int i = 0; i < e.nflags; i++) e.flags[i * e.flag_stride] |= 1ull << (e.x >> 6);
    if (e.value >= 4u) *e.reserved = 1u;
    const u32 code = (e.value >= 4u ? (u32)FS3D_STATIC : e.value) ^ 1u;
    u32 *w = e.planes + 4 * e.word + (e.x & 1);
    const u32 m = 1u << pair_bit((e.x & 63) >> 1);
    w[0] = (code & 1u) ? w[0] | m : w[0] & ~m;
    w[2] = (code & 2u) ? w[2] | m : w[2] & ~m;
  }
  post_note(n, 0);
}

__global__ void post_byte_kernel(const u8 *p, Note n) {
  if (threadIdx.x == 0) post_note(n, *p);
}

__global__ void post_kernel(const u64 *p, Note n) {
  if (threadIdx.x == 0) post_note(n, *p);
}

// Four cells per lane: a lane's chain of mixes, not their number, is what takes the
// time.  Workgroups add to one word, and the last one posts the sum (hash_parts[0],
// and the count beside it, are 0 between launches).  48 x 37 x 29, hashed after a tick:
// 14 us for a tick that hashes as it writes, the sum of its parts and the note, 9 for
// a tick and this.
__global__ __launch_bounds__(256) void hash_post_kernel(const u8 *g, u32 n, u64 *parts, Note note) {
  const u32 i = 4u * (blockIdx.x * 256u + threadIdx.x);
  u64 acc = 0;
  if (i < n) {
    const u32 d = *reinterpret_cast<const u32 *>(g + i);
#pragma unroll
    for (u32 k = 0; k < 4; k++) {
      const u32 v = (d >> (8 * k)) & 0xFFu;
      if (i + k < n && v) acc += planedev::dmix64(((u64)(i + k) << 8) | v);
    }
  }
  __shared__ u64 wsum[4];
  acc = planedev::wave_sum_u64(acc);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x != 0) return;
  atomicAdd((unsigned long long *)parts, (unsigned long long)(wsum[0] + wsum[1] + wsum[2] + wsum[3]));
  __threadfence();
  if (atomicAdd((unsigned long long *)parts + 1, 1ull) != gridDim.x - 1ull) return;
  __threadfence();
  const u64 sum = atomicExch((unsigned long long *)parts, 0ull);
  atomicExch((unsigned long long *)parts + 1, 0ull);
  post_note(note, sum);
}

}  // namespace

hipError_t launch_hash_post(const u8 *g, size_t n, u64 *hash_parts, const Note &note, hipStream_t s) {
  hipLaunchKernelGGL(hash_post_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, g, (u32)n, hash_parts,
                     note);
  return hipGetLastError();
}

hipError_t launch_set_cell(const CellEdit &e, const Note &n, hipStream_t s) {
  hipLaunchKernelGGL(set_cell_kernel, dim3(1), dim3(64), 0, s, e, n);
  return hipGetLastError();
}

hipError_t launch_post_byte(const u8 *p, const Note &n, hipStream_t s) {
  hipLaunchKernelGGL(post_byte_kernel, dim3(1), dim3(64), 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_post(const u64 *p, const Note &n, hipStream_t s) {
  hipLaunchKernelGGL(post_kernel, dim3(1), dim3(64), 0, s, p, n);
  return hipGetLastError();
}

}  // namespace fs3d
