// Copies from device memory to pageable host memory through pinned staging slots.
//
// Left to the runtime, such a copy is one thread moving pieces through a staging
// buffer: 18 GB/s into pages that exist and 11 GB/s into fresh ones, which that
// thread also has to fault in, where the link carries 56 GB/s.  Here a kernel writes
// the bytes to pinned slots, a launch to as many as are free, and up to four threads
// copy out of the slots (copy_job.h), so that the link, the copying and the page faults
// overlap.
// A piece reports itself by a flag in pinned memory: a copy command per piece takes
// 10 us more than its bytes, an event 5.  Only the calling thread talks to the
// runtime, whose first call in a new thread costs 100 us and more.
// (The other direction is left to the runtime, which pins the pages and reads them in
// place: 134 MB in 4.5 ms.)
#include "hostcopy.h"

#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>

#include "copy_job.h"

namespace fs3d {
namespace {

typedef u32 u32x4 __attribute__((ext_vector_type(4)));

constexpr size_t kSlots = kCopySlots;
constexpr size_t kSlotBytes = 1u << 20;
constexpr size_t kAloneMax = 512u << 10;  // up to here the calling thread copies alone
constexpr size_t kDirectMax = 64u << 10;  // below, the runtime's copy is as fast

// src 16-byte aligned.
__global__ __launch_bounds__(256) void piece_kernel(const u8 *src, PieceOut o) {
  const PinnedOut out(o.buf, o.n);
  const u32 base = blockIdx.x * kBlockBytes, words = o.n / 16u, first = base / 16u + threadIdx.x;
  u32x4 v[kBlockBytes / 4096];
#pragma unroll
  for (u32 k = 0; k < kBlockBytes / 4096; k++)
    if (first + 256u * k < words) v[k] = reinterpret_cast<const u32x4 *>(src)[first + 256u * k];
#pragma unroll
  for (u32 k = 0; k < kBlockBytes / 4096; k++)
    if (first + 256u * k < words) out.store16(16u * (first + 256u * k), v[k]);
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x < o.n % 16u)
    out.store1(16u * words + threadIdx.x, src[16u * words + threadIdx.x]);
  piece_done(o);
}

constexpr size_t kFlagBytes = kSlots * kFlagStride * sizeof(u32);

struct Staging {
  int dev = 0;
  size_t bytes = 0;         // of the slots
  u8 *mem = nullptr;        // a flag for each slot, then the slots
  u32 *counters = nullptr;  // device memory, one per slot
  bool cleared = false;     // the counters have been set to 0
  hipStream_t stream = nullptr;  // for work that has no stream of its own, once there was some
  u32 *flag(size_t k) const { return reinterpret_cast<u32 *>(mem) + kFlagStride * k; }
  u8 *slots() const { return mem + kFlagBytes; }
};

void destroy(Staging *g) {
  if (!g) return;
  if (g->stream) (void)hipStreamDestroy(g->stream);
  if (g->counters) (void)hipFree(g->counters);
  if (g->mem) (void)hipHostFree(g->mem);
  delete g;
}

// Slots for a copy of `total` bytes: a small copy's are made in a tenth of a
// millisecond, all twelve in a fifth.
Staging *create(int dev, size_t total) {
  Staging *g = new (std::nothrow) Staging();
  if (!g) return nullptr;
  g->dev = dev;
  g->bytes = std::min(kSlots * kSlotBytes, std::max(total, (size_t)1 << 20));
  hipError_t e = hipHostMalloc((void **)&g->mem, kFlagBytes + g->bytes, hipHostMallocDefault);
  if (e == hipSuccess) e = hipMalloc((void **)&g->counters, kSlots * sizeof(u32));
  if (e == hipSuccess) return g;
  (void)hipGetLastError();
  destroy(g);
  return nullptr;
}

// One idle staging is kept (12 MiB at most); every copy in flight has its own.
std::mutex g_mutex;
Staging *g_idle = nullptr;
int g_worlds = 0;

Staging *acquire(int dev, size_t total) {
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_idle && g_idle->dev == dev && g_idle->bytes >= std::min(total, kSlots * kSlotBytes)) {
      Staging *g = g_idle;
      g_idle = nullptr;
      return g;
    }
  }
  return create(dev, total);
}

void give_back(Staging *g) {
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    std::swap(g, g_idle);
  }
  destroy(g);
}

// Launches the kernel for bytes [off, off + out.n) of a span.
typedef std::function<hipError_t(size_t span, size_t off, const PieceOut &out, hipStream_t)> Issue;

CopyHelpers g_helpers;

// The launches of a copy through g's slots.
struct Slots {
  Staging *g;
  size_t piece;
  hipStream_t s;
  const Issue &make;
  int issue(const CopyPiece &p, size_t slot, size_t bytes, u32 value) const {
    return make(p.span, p.off,
                PieceOut{g->slots() + slot * piece, (u32)bytes, (u32)piece, g->counters + slot, g->flag(slot), value},
                s);
  }
  int wait() const { return hipStreamSynchronize(s); }
  int lost() const { return hipErrorUnknown; }
};

// Runs the pieces through g; the stream is idle when it returns.
hipError_t run(Staging *g, std::vector<CopyPiece> pieces, size_t piece, size_t total, hipStream_t s,
               const Issue &issue) {
  const std::shared_ptr<CopyJob> job = std::make_shared<CopyJob>();
  job->pieces = std::move(pieces);
  job->mem = g->slots();
  job->flags = g->flag(0);
  job->flag_stride = kFlagStride;
  job->piece = piece;
  job->slots = std::min(kSlots, g->bytes / piece);
  for (size_t k = 0; k < kSlots; k++) *g->flag(k) = 0;
  if (!g->cleared)
    if (const hipError_t e = launch_fill_u32(g->counters, kSlots, 0, s)) return e;
  const int helpers = total > kAloneMax ? (int)std::min<size_t>(CopyHelpers::kMost, job->pieces.size() - 1) : 0;
  const hipError_t e = (hipError_t)copy_run(job, &g_helpers, helpers, Slots{g, piece, s, issue});
  g->cleared = e == hipSuccess;  // (a launch that failed may have left counts)
  return e;
}

void split(std::vector<CopyPiece> *pieces, void *host, size_t n, size_t span, size_t piece) {
  for (size_t off = 0; off < n; off += piece)
    pieces->push_back(CopyPiece{(u8 *)host + off, off, std::min(piece, n - off), span});
}

// The first piece of a small copy is there soon, and no helper is left without one.
size_t piece_of(size_t total) {
  return std::min(kSlotBytes, std::max<size_t>(kDirectMax, (total / 16 + kBlockBytes - 1) / kBlockBytes * kBlockBytes));
}

// Memory that the runtime knows (pinned, managed, of a device) it copies directly.
bool pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t copy_to_host(const std::vector<HostSpan> &spans, int dev, hipStream_t s) {
  size_t total = 0;
  bool staged = true;
  for (const HostSpan &h : spans) {
    total += h.n;
    staged = staged && pageable(h.host) && (uintptr_t)h.dev % 16 == 0;
  }
  Staging *g = staged && total >= kDirectMax ? acquire(dev, total) : nullptr;
  if (!g) {
    for (const HostSpan &h : spans)
      if (const hipError_t e = hipMemcpyAsync(h.host, h.dev, h.n, hipMemcpyDeviceToHost, s)) return e;
    return hipStreamSynchronize(s);
  }
  hipError_t e = hipErrorOutOfMemory;
  try {
    std::vector<CopyPiece> pieces;
    for (size_t i = 0; i < spans.size(); i++) split(&pieces, spans[i].host, spans[i].n, i, piece_of(total));
    e = run(g, pieces, piece_of(total), total, s, [&](size_t i, size_t off, const PieceOut &out, hipStream_t st) {
      hipLaunchKernelGGL(piece_kernel, dim3(piece_blocks(out)), dim3(256), 0, st, (const u8 *)spans[i].dev + off, out);
      return hipGetLastError();
    });
  } catch (...) {
    e = hipErrorOutOfMemory;
  }
  give_back(g);
  return e;
}

hipError_t make_on_host(void *host, size_t n, int dev,
                        const std::function<hipError_t(size_t, const PieceOut &, hipStream_t)> &make) {
  Staging *g = acquire(dev, n);
  if (!g) return hipErrorOutOfMemory;
  hipError_t e = hipErrorOutOfMemory;
  try {
    std::vector<u8> between;  // the threads write ordinary memory only
    if (!pageable(host)) between.resize(n);
    std::vector<CopyPiece> pieces;
    split(&pieces, between.empty() ? host : between.data(), n, 0, piece_of(n));
    e = g->stream ? hipSuccess : hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking);
    if (e == hipSuccess)
      e = run(g, pieces, piece_of(n), n, g->stream,
              [&](size_t, size_t off, const PieceOut &out, hipStream_t st) { return make(off, out, st); });
    if (e == hipSuccess && !between.empty()) e = hipMemcpy(host, between.data(), n, hipMemcpyDefault);
  } catch (...) {
    e = hipErrorOutOfMemory;
  }
  give_back(g);
  return e;
}

void hostcopy_world(int delta) {
  Staging *g = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_worlds += delta;
    if (g_worlds == 0) std::swap(g, g_idle);
  }
  destroy(g);
}

}  // namespace fs3d
