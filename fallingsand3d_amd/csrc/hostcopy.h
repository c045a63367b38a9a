// Copies from device memory to ordinary (pageable) host memory.
#pragma once

#include <functional>
#include <vector>

#include "fs3d_internal.h"

namespace fs3d {

struct HostSpan {
  void *host;
  const void *dev;
  size_t n;
};

// A buffer of pinned host memory.  Stores go through the caches to the memory (scope
// bits SC0 | SC1), so that waiting for them is all it takes to hand them to the host:
// writing the caches back in every workgroup instead halved the rate of the link.
struct PinnedOut {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ PinnedOut(void *p, u32 bytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00020000)) {}
  template <typename V>
  __device__ __forceinline__ void store16(u32 off, V v) const {
    typedef u32 u32x4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rsrc, (int)off, 0, kThrough);
  }
  __device__ __forceinline__ void store1(u32 off, u8 v) const {
    __builtin_amdgcn_raw_buffer_store_b8(v, rsrc, (int)off, 0, kThrough);
  }
  static constexpr int kThrough = 1 | 16;
};

// What one launch writes: n bytes at buf, in pieces of `piece` bytes (a multiple of
// kBlockBytes).  The last workgroup of piece i to finish stores value + i to its flag.
struct PieceOut {
  u8 *buf;
  u32 n, piece;
  u32 *counters;  // device memory, one per piece, 0 between launches
  u32 *flags;     // pinned, kFlagStride apart
  u32 value;
};
constexpr u32 kBlockBytes = 16384;  // written by a workgroup of 256
constexpr u32 kFlagStride = 16;

inline unsigned piece_blocks(const PieceOut &o) { return (o.n + kBlockBytes - 1) / kBlockBytes; }

// Called by whole workgroups, after their last PinnedOut store.
__device__ __forceinline__ void piece_done(const PieceOut &o) {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // this wave's stores are in memory (vmcnt 0)
  __syncthreads();
  if (threadIdx.x == 0) {
    const u32 i = blockIdx.x * kBlockBytes / o.piece;
    const u32 bytes = min(o.piece, o.n - i * o.piece);
    if (atomicAdd(o.counters + i, 1u) == (bytes + kBlockBytes - 1) / kBlockBytes - 1u) {
      o.counters[i] = 0;
      __hip_atomic_store(o.flags + i * kFlagStride, o.value + i, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// Copies dev to host after the work already in stream s; done when it returns.
hipError_t copy_to_host(const std::vector<HostSpan> &spans, int dev, hipStream_t s);
// n bytes made on the device: make(off, out, stream) launches one kernel of
// piece_blocks(out) workgroups that writes bytes [off, off + out.n).
hipError_t make_on_host(void *host, size_t n, int dev,
                        const std::function<hipError_t(size_t, const PieceOut &, hipStream_t)> &make);

// Worlds alive: the staging memory kept for the next copy goes with the last one.
void hostcopy_world(int delta);

}  // namespace fs3d
