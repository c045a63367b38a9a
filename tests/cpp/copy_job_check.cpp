// The threads that copy out of staging slots (copy_job.h), with a thread in place of the
// device: every byte of several spans, copies in several threads at once, a device that is
// busy with something else for long, launches that fail, pieces that never come, and
// helpers that are gone when their owner is.
#include <condition_variable>
#include <cstdio>
#include <ctime>
#include <deque>
#include <dirent.h>
#include <random>

#include "../../fallingsand3d_amd/csrc/copy_job.h"

using namespace fs3d;

#define CHECK(c)                                         \
  do {                                                   \
    if (!(c)) {                                          \
      std::printf("FAILED line %d: %s\n", __LINE__, #c); \
      return 1;                                          \
    }                                                    \
  } while (0)

// Fills slots in order, like a stream; the first launch waits for `ahead` ms of other work.
struct Device {
  struct Launch {
    const uint8_t *src;
    size_t slot, bytes;
    uint32_t value;
  };
  std::vector<std::vector<uint8_t>> spans;
  std::vector<uint8_t> mem;
  std::vector<uint32_t> flags = std::vector<uint32_t>(kCopySlots, 0);
  size_t piece;
  int ahead = 0, fail_at = -1, lose_at = -1, launches = 0;
  std::mutex m;
  std::condition_variable cv, idle;
  std::deque<Launch> queue;
  bool end = false, running = false;
  std::thread thread;

  explicit Device(size_t piece_bytes) : mem(piece_bytes * kCopySlots), piece(piece_bytes) {
    thread = std::thread([this] { work(); });
  }
  ~Device() {
    {
      std::lock_guard<std::mutex> l(m);
      end = true;
    }
    cv.notify_all();
    thread.join();
  }
  void work() {
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      cv.wait(l, [&] { return end || !queue.empty(); });
      if (queue.empty()) return;
      const Launch a = queue.front();
      queue.pop_front();
      running = true;
      const int ms = ahead;
      ahead = 0;
      l.unlock();
      if (ms) std::this_thread::sleep_for(std::chrono::milliseconds(ms));
      for (size_t i = 0, off = 0; off < a.bytes; i++, off += piece) {
        const size_t n = std::min(piece, a.bytes - off);
        std::memcpy(mem.data() + (a.slot + i) * piece, a.src + off, n);
        if ((int)(a.value + i) - 1 != lose_at) __atomic_store_n(&flags[a.slot + i], a.value + (uint32_t)i, __ATOMIC_RELEASE);
      }
      l.lock();
      running = false;
      if (queue.empty()) idle.notify_all();
    }
  }
  struct Calls {
    Device *d;
    int issue(const CopyPiece &p, size_t slot, size_t bytes, uint32_t value) const {
      if (d->launches++ == d->fail_at) return 7;
      std::lock_guard<std::mutex> l(d->m);
      d->queue.push_back({d->spans[p.span].data() + p.off, slot, bytes, value});
      d->cv.notify_all();
      return 0;
    }
    int wait() const {
      std::unique_lock<std::mutex> l(d->m);
      d->idle.wait(l, [&] { return d->queue.empty() && !d->running; });
      return 0;
    }
    int lost() const { return 9; }
  };
};

static std::atomic<double> cpu_seconds{0};  // of the last copy, all threads

static int copy(Device *d, CopyHelpers *helpers, int n_helpers, size_t slots, const std::vector<size_t> &sizes,
                unsigned seed, bool *right) {
  std::mt19937 rng(seed);
  d->spans.clear();
  std::vector<std::vector<uint8_t>> out;
  auto job = std::make_shared<CopyJob>();
  for (size_t i = 0; i < sizes.size(); i++) {
    d->spans.emplace_back(sizes[i]);
    for (uint8_t &b : d->spans.back()) b = (uint8_t)rng();
    out.emplace_back(sizes[i], (uint8_t)0);
  }
  for (size_t i = 0; i < sizes.size(); i++)
    for (size_t off = 0; off < sizes[i]; off += d->piece)
      job->pieces.push_back(CopyPiece{out[i].data() + off, off, std::min(d->piece, sizes[i] - off), i});
  job->mem = d->mem.data();
  job->flags = d->flags.data();
  job->flag_stride = 1;
  job->piece = d->piece;
  job->slots = slots;
  for (uint32_t &f : d->flags) f = 0;
  const std::clock_t c0 = std::clock();
  const int e = copy_run(job, helpers, n_helpers, Device::Calls{d});
  cpu_seconds = (double)(std::clock() - c0) / CLOCKS_PER_SEC;
  *right = out == d->spans;
  return e;
}

static int threads_alive() {
  int n = 0;
  if (DIR *dir = opendir("/proc/self/task")) {
    while (dirent *e = readdir(dir)) n += e->d_name[0] != '.';
    closedir(dir);
  }
  return n;
}

static int right_bytes() {
  CopyHelpers helpers;
  Device d(1000);
  bool right = false;
  for (unsigned k = 0; k < 60; k++) {
    const std::vector<size_t> sizes = {1 + 977 * k, 1 + (k * 31) % 50, 3 * k * k + 1};
    CHECK(copy(&d, &helpers, (int)(k % 4), 1 + k % kCopySlots, sizes, k, &right) == 0 && right);
  }
  return 0;
}

static int many_threads() {
  CopyHelpers helpers;
  std::atomic<int> bad{0};
  std::vector<std::thread> ts;
  for (unsigned i = 0; i < 4; i++)
    ts.emplace_back([&, i] {
      Device d(4096);
      for (unsigned k = 0; k < 12; k++) {
        bool right = false;
        if (copy(&d, &helpers, 3, kCopySlots, {300000 + i, 5000}, i * 100 + k, &right) || !right) bad++;
      }
    });
  for (std::thread &t : ts) t.join();
  CHECK(bad == 0);
  return 0;
}

// 400 ms of other work ahead: nobody spins through it.
[[maybe_unused]] static int long_wait() {
  CopyHelpers helpers;
  Device d(65536);
  d.ahead = 400;
  bool right = false;
  const auto t0 = std::chrono::steady_clock::now();
  CHECK(copy(&d, &helpers, 3, kCopySlots, {65536 * 15}, 1, &right) == 0 && right);
  const double cpu = cpu_seconds;
  const double wall = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  std::printf("%.0f ms on the clock, %.0f ms of processor time\n", wall * 1e3, cpu * 1e3);
  CHECK(wall > 0.4 && cpu < 0.25 * wall);
  return 0;
}

static int failures() {
  CopyHelpers helpers;
  bool right = true;
  for (int at = 0; at < 3; at++) {
    Device a(1000);
    a.fail_at = at;
    CHECK(copy(&a, &helpers, 3, 4, {20000}, 1, &right) == 7 && !right);
    for (int lost = 0; lost < 20; lost += 3) {  // found by whoever has claimed it
      Device b(1000);
      b.lose_at = lost;
      CHECK(copy(&b, &helpers, at, 4, {20000}, 1, &right) == 9 && !right);
    }
  }
  return 0;
}

static int gone(int at_start) {
  {
    CopyHelpers helpers;
    {
      Device d(1000);
      bool right = false;
      for (unsigned k = 0; k < 20; k++) CHECK(copy(&d, &helpers, 3, kCopySlots, {3000}, k, &right) == 0 && right);
    }
    CHECK(threads_alive() > at_start);
  }
  // (a thread that has been joined may still be listed for a moment)
  for (int k = 0; k < 1000 && threads_alive() > at_start; k++)
    std::this_thread::sleep_for(std::chrono::milliseconds(1));
  CHECK(threads_alive() == at_start);
  return 0;
}

int main() {
  // (a sanitizer has a thread of its own, from the first one on)
  std::thread([] {}).join();
  int at_start = threads_alive();
  for (int k = 0; k < 50; k++) {
    std::this_thread::sleep_for(std::chrono::milliseconds(1));
    at_start = std::min(at_start, threads_alive());
  }
  if (right_bytes() || many_threads() || failures() || gone(at_start)) return 1;
#ifndef __SANITIZE_THREAD__
  if (long_wait()) return 1;
#endif
  std::printf("copy job checks passed\n");
  return 0;
}
