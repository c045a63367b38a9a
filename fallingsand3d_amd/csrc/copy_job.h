// Copying out of staging slots that a device fills: the calling thread and a few helpers
// share a job's pieces.  Host code without device calls, which are the caller's (Dev).
#pragma once

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <deque>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace fs3d {

constexpr size_t kCopySlots = 12;

struct CopyPiece {
  uint8_t *host;
  size_t off, n;  // in its span
  size_t span;
};

// Piece c goes through slot c % slots; the slot's flag becomes c + 1 when it is there.
// A helper that gets to run only after the copy is over finds nothing to claim and touches
// nothing but the job, so that the copy does not wait for it.  (Waited for, helpers that
// were not scheduled for a while made a copy of 0.3 ms take 4.)
struct CopyJob {
  std::vector<CopyPiece> pieces;
  const uint8_t *mem = nullptr;  // the slots
  const uint32_t *flags = nullptr;
  size_t flag_stride = 0;
  size_t piece = 0, slots = 0;                 // bytes of a slot, slots in use
  std::atomic<size_t> taken{0};                // pieces claimed
  std::atomic<size_t> copied{0};               // pieces copied out
  std::atomic<int> busy{0};                    // helpers between a claim and its end
  std::atomic<size_t> done[kCopySlots] = {};   // of a slot: the last piece copied out of it, plus 1
  std::atomic<bool> stop{false};

  bool arrived(size_t c) const {
    return __atomic_load_n(flags + (c % slots) * flag_stride, __ATOMIC_ACQUIRE) == (uint32_t)c + 1u;
  }
  void copy_out(size_t c) {
    const CopyPiece &p = pieces[c];
    std::memcpy(p.host, mem + (c % slots) * piece, p.n);
    done[c % slots].store(c + 1, std::memory_order_release);
    copied.fetch_add(1);
  }
};

// How a thread waits: it looks again and again for the time that a frame and the pieces of a
// copy take, then sleeps in between, the longer the longer it has waited, since what is
// ahead in the stream may take any time.  (Twelve slots take 0.2 ms to fill, which is about
// when the first of them is there: asleep from then on, 33 MB took 870 us instead of 790.)
class Patience {
 public:
  bool spent() const { return waited() > std::chrono::milliseconds(2); }
  void wait() const {
    if (!spent()) return std::this_thread::yield();
    const auto most = std::chrono::milliseconds(2);
    const auto part = waited() / 4;
    std::this_thread::sleep_for(part < most ? part : most);
  }

 private:
  std::chrono::nanoseconds waited() const { return std::chrono::steady_clock::now() - start_; }
  std::chrono::steady_clock::time_point start_ = std::chrono::steady_clock::now();
};

inline void copy_help(CopyJob *j) {
  for (;;) {
    j->busy.fetch_add(1);
    const size_t c = j->stop.load() ? j->pieces.size() : j->taken.fetch_add(1);
    bool mine = c < j->pieces.size();
    for (const Patience p; mine && !j->arrived(c);) {
      if (j->stop.load()) mine = false;
      p.wait();
    }
    if (mine) j->copy_out(c);
    j->busy.fetch_sub(1);
    if (!mine) return;
  }
}

// The helper threads: a few that sleep between copies, made by the first one.  They run
// this code until their owner is gone, which waits for them.
class CopyHelpers {
 public:
  static constexpr int kMost = 3;  // (11 were no faster)

  ~CopyHelpers() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      end_ = true;
      for (auto &j : running_) j->stop.store(true);
    }
    wake_.notify_all();
    if (pid_ == getpid())
      for (std::thread &t : threads_) t.join();
    else  // forked: the threads are not in this process
      for (std::thread &t : threads_) t.detach();
  }
  // Lets up to n of them help with the job, as they become free.
  void start(int n, const std::shared_ptr<CopyJob> &job) {
    std::lock_guard<std::mutex> lock(mutex_);
    try {
      if (pid_ != getpid()) {
        for (std::thread &t : threads_) t.detach();
        threads_.clear();
        pid_ = getpid();
      }
      threads_.reserve(kMost);
      while ((int)threads_.size() < kMost) threads_.emplace_back([this] { work(); });
    } catch (...) {
      // fewer threads do the same work
    }
    for (int i = 0; i < n && i < (int)threads_.size(); i++) {
      waiting_.push_back(job);
      wake_.notify_one();
    }
  }
  // The job is over: who has not begun to help need not.
  void forget(const std::shared_ptr<CopyJob> &job) {
    std::lock_guard<std::mutex> lock(mutex_);
    waiting_.erase(std::remove(waiting_.begin(), waiting_.end(), job), waiting_.end());
  }

 private:
  void work() {
    std::unique_lock<std::mutex> lock(mutex_);
    for (;;) {
      wake_.wait(lock, [this] { return end_ || !waiting_.empty(); });
      if (end_) return;
      const std::shared_ptr<CopyJob> job = waiting_.front();
      waiting_.pop_front();
      running_.push_back(job);
      lock.unlock();
      copy_help(job.get());
      lock.lock();
      running_.erase(std::find(running_.begin(), running_.end(), job));
    }
  }
  std::mutex mutex_;
  std::condition_variable wake_;
  std::deque<std::shared_ptr<CopyJob>> waiting_;
  std::vector<std::shared_ptr<CopyJob>> running_;
  std::vector<std::thread> threads_;
  pid_t pid_ = getpid();
  bool end_ = false;
};

// Runs the job with up to `helpers` helper threads; 0 or dev's first error.  Dev:
//   issue(piece, slot, bytes, value)  launches what fills the slots from `slot` on with
//                                     `bytes` bytes from the piece on; the first slot's flag
//                                     becomes value, the next one's value + 1 ...
//   wait()                            until what was launched has ended
//   lost()                            the error of a piece that is not there after that
// Nothing launched is running when it returns.
template <class Dev>
int copy_run(const std::shared_ptr<CopyJob> &job, CopyHelpers *threads, int helpers, Dev &&dev) {
  CopyJob &j = *job;
  const std::vector<CopyPiece> &pieces = j.pieces;
  const size_t n = pieces.size(), slots = j.slots;
  size_t issued = 0;
  int e = 0;
  // Launches what follows in free neighbouring slots (once a few are free).
  auto issue_free = [&] {
    while (issued < n && e == 0) {
      const CopyPiece &p = pieces[issued];
      size_t m = 0, bytes = 0;
      while (issued + m < n && pieces[issued + m].span == p.span && issued % slots + m < slots &&
             (issued + m < slots ||
              j.done[issued % slots + m].load(std::memory_order_acquire) == issued + m - slots + 1)) {
        bytes += pieces[issued + m].n;
        m++;
      }
      const bool all = issued + m == n || issued % slots + m == slots || pieces[issued + m].span != p.span;
      if (m == 0 || (m < slots / 4 && !all)) return;
      e = dev.issue(p, issued % slots, bytes, (uint32_t)issued + 1u);
      issued += m;
    }
  };
  issue_free();
  if (helpers > 0) threads->start(helpers, job);
  // Waits a little.  What the threads wait for ends with its launch: once those have ended,
  // a piece whose flag is not there, whoever has claimed it, is lost.
  size_t ended = 0;
  auto wait_on = [&](const Patience &p) {
    if (!p.spent() || ended == issued) return p.wait();
    e = dev.wait();
    ended = issued;
    for (size_t c = issued > slots ? issued - slots : 0; c < issued && !e; c++)
      if (j.done[c % slots].load(std::memory_order_acquire) != c + 1 && !j.arrived(c)) e = dev.lost();
  };
  // The calling thread issues the pieces and copies too.
  while (e == 0) {
    const size_t c = j.taken.fetch_add(1);
    if (c >= n && issued == n) break;
    for (const Patience p;;) {
      issue_free();
      if (e || (c >= n ? issued == n : c < issued && j.arrived(c))) break;
      wait_on(p);
    }
    if (e == 0 && c < n) j.copy_out(c);
  }
  for (const Patience p; e == 0 && j.copied.load() < n;) wait_on(p);
  if (e != 0) j.stop.store(true);
  for (const Patience p; e != 0 && j.busy.load() != 0;) p.wait();
  if (helpers > 0) threads->forget(job);
  const int last = dev.wait();
  return e ? e : last;
}

}  // namespace fs3d
