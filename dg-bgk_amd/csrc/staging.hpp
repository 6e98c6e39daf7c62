// staging.hpp -- host <-> device transfers of the caller's (pageable) arrays
// through pinned blocks.
//
// A pageable copy of tens of megabytes is bound by one host thread: 30 GB/s
// to the device, 18 GB/s back, less where the caller's array is touched for
// the first time, against 57 GB/s over the bus from pinned memory.  Here up
// to kWorkers threads move pieces between the array and pinned blocks while
// the bus carries others.  Small arrays go through one pinned block on the
// calling thread (a pageable copy of a few KB costs a blit kernel and a wait
// of its own).
//
// The blocks belong to the process: at most kKeep stay in the pool, handed out
// under a lock to any thread and given back idle, and all are freed when the
// last context is destroyed.  Nothing here allocates on the heap but the
// threads, so no entry point throws.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>

namespace dgbgk {

constexpr size_t kStageBlock = (size_t)2 << 20;
// f of 26,237 triangles x 128 to the device, a step, and back into a fresh
// array (81 MB each way): 9.4 ms with one thread, 6.4 with two, 5.3 with
// three, 4.9 with four (11.7 pageable).
constexpr int kWorkers = 4;
// To the device, from arrays up to this size, the runtime's own pageable copy
// (27 GB/s at 3 MB, 38 at 32 MB): the workers' threads and blocks cost more
// than they gain.  set_f, ms, with them -> without: 3.2 MB 0.18 -> 0.15, 8 MB
// 0.36 -> 0.29, 27 MB 0.86 -> 0.82, but 52 MB (past the host's cache) 1.55 ->
// 1.98.
constexpr size_t kPageableIn = (size_t)32 << 20;

class StagePool {
 public:
  static StagePool& get() {
    static StagePool p;
    return p;
  }
  void user(int d) {  // +1 / -1: a context begins / ends
    std::lock_guard<std::mutex> l(mu_);
    users_ += d;
    if (users_ > 0) return;
    while (n_) (void)hipHostFree(free_[--n_]);
  }
  char* take() {
    {
      std::lock_guard<std::mutex> l(mu_);
      if (n_) return free_[--n_];
    }
    void* b = nullptr;
    // portable: usable with every device
    if (hipHostMalloc(&b, kStageBlock, hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();  // the caller falls back to a pageable copy
      return nullptr;
    }
    return (char*)b;
  }
  void give(char* b) {
    if (!b) return;
    {
      std::lock_guard<std::mutex> l(mu_);
      if (users_ > 0 && n_ < kKeep) {
        free_[n_++] = b;
        return;
      }
    }
    (void)hipHostFree(b);
  }

 private:
  static constexpr int kKeep = 4 * kWorkers;
  std::mutex mu_;
  char* free_[kKeep];
  int n_ = 0;
  int users_ = 0;
};

// A pinned block for the scope (p null if none could be had), with the copies
// a stream carries to or from it.  It goes back idle on every way out of the
// scope: one that a copy may still use, and whose stream cannot be waited
// for, is not handed out again.
class StageBlock {
 public:
  char* const p;
  explicit StageBlock(hipStream_t s, bool wanted = true)
      : p(wanted ? StagePool::get().take() : nullptr), s_(s) {}
  ~StageBlock() {
    if (!busy_ || hipStreamSynchronize(s_) == hipSuccess) StagePool::get().give(p);
  }
  StageBlock(const StageBlock&) = delete;
  StageBlock& operator=(const StageBlock&) = delete;
  hipError_t copy(void* to, const void* from, size_t n, hipMemcpyKind kind) {
    busy_ = true;
    return hipMemcpyAsync(to, from, n, kind, s_);
  }
  hipError_t wait() {
    const hipError_t e = hipStreamSynchronize(s_);
    busy_ = busy_ && e != hipSuccess;
    return e;
  }

 private:
  const hipStream_t s_;
  bool busy_ = false;
};

// fn(w) for w < n (at most kWorkers), on this thread and n - 1 others that
// begin on the same device.  Where no thread can be had, in turn.
template <typename F>
void on_workers(int n, int dev, F fn) {
  std::thread t[kWorkers];
  int w = 1;
  try {
    for (; w < n; ++w)
      t[w] = std::thread([&, w] {
        if (hipSetDevice(dev) == hipSuccess) fn(w);
      });
  } catch (...) {
  }
  fn(0);
  for (int r = w; r < n; ++r) fn(r);
  for (auto& x : t)
    if (x.joinable()) x.join();
}

// Small results: device ranges to as many arrays of the caller's (host null:
// not wanted), at most a block in all, adjacent ranges as one copy.  In order
// after the work on the stream; the data has arrived, and nothing writes to
// the arrays any more, on return.
struct StagePart {
  const void* dev;
  void* host;
  size_t n;
};
inline hipError_t stage_fetch(const StagePart* part, int parts, hipStream_t stream) {
  StageBlock b(stream);
  hipError_t e = hipSuccess;
  size_t at = 0;
  for (int i = 0, j; i < parts && e == hipSuccess; i = j) {
    size_t n = part[i].n;
    for (j = i + 1; b.p && j < parts && part[j].dev == (const char*)part[i].dev + n; ++j)
      n += part[j].n;
    if (b.p)
      e = b.copy(b.p + at, part[i].dev, n, hipMemcpyDeviceToHost);
    else if (part[i].host)
      e = b.copy(part[i].host, part[i].dev, n, hipMemcpyDeviceToHost);
    at += n;
  }
  const hipError_t f = b.wait();
  if (e == hipSuccess) e = f;
  at = 0;
  for (int i = 0; e == hipSuccess && b.p && i < parts; at += part[i++].n)
    if (part[i].host) std::memcpy(part[i].host, b.p + at, part[i].n);
  return e;
}

// Copies n bytes between the caller's array and device memory, in order
// after the work on the stream, and returns when the data has arrived.
// toDev: host is read, else written.  whole: the size of the array this is a
// part of, if larger.
inline hipError_t stage_copy(void* dev, void* host, size_t n, bool toDev, hipStream_t stream,
                             int device, size_t whole = 0) {
  const hipMemcpyKind kind = toDev ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
  auto plain = [&](char* d, char* h, size_t m) {
    hipError_t e = toDev ? hipMemcpyAsync(d, h, m, kind, stream) : hipMemcpyAsync(h, d, m, kind, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  };
  const size_t pieces = (n + kStageBlock - 1) / kStageBlock;
  if (!n) return hipSuccess;
  if (pieces == 1) {
    StageBlock b(stream);
    if (!b.p) return plain((char*)dev, (char*)host, n);
    if (toDev) std::memcpy(b.p, host, n);
    hipError_t e = toDev ? b.copy(dev, b.p, n, kind) : b.copy(b.p, dev, n, kind);
    if (e == hipSuccess) e = b.wait();
    if (e == hipSuccess && !toDev) std::memcpy(host, b.p, n);
    return e;
  }
  if (toDev && std::max(n, whole) <= kPageableIn) return plain((char*)dev, (char*)host, n);
  // each worker takes pieces w, w + workers, ... through two blocks: one on
  // the bus while the other is filled or emptied
  const int workers = (int)std::min<size_t>(kWorkers, pieces);
  hipError_t err[kWorkers];
  std::fill(err, err + workers, hipErrorInvalidDevice);  // a worker that never began
  on_workers(workers, device, [&](int w) {
    const bool both = (size_t)(w + workers) < pieces;
    StageBlock b[2] = {StageBlock(stream), StageBlock(stream, both)};
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipError_t e = hipSuccess;
    auto ok = [&](hipError_t x) { return (e = x) == hipSuccess; };
    auto at = [&](size_t i) { return i * kStageBlock; };
    auto len = [&](size_t i) { return std::min(kStageBlock, n - at(i)); };
    const bool staged = b[0].p && (!both || b[1].p) &&
                        hipEventCreateWithFlags(&ev[0], hipEventDisableTiming) == hipSuccess &&
                        hipEventCreateWithFlags(&ev[1], hipEventDisableTiming) == hipSuccess;
    char *d = (char*)dev, *h = (char*)host;
    size_t i = w;
    if (!staged) {
      (void)hipGetLastError();
      for (; i < pieces && ok(plain(d + at(i), h + at(i), len(i))); i += workers) {
      }
    } else if (toDev) {
      for (int k = 0; i < pieces; i += workers, ++k) {
        const int s = k & 1;
        if (k >= 2 && !ok(hipEventSynchronize(ev[s]))) break;
        std::memcpy(b[s].p, h + at(i), len(i));
        if (!ok(b[s].copy(d + at(i), b[s].p, len(i), kind))) break;
        if (!ok(hipEventRecord(ev[s], stream))) break;
      }
    } else {
      auto fetch = [&](size_t j, int s) {
        return ok(b[s].copy(b[s].p, d + at(j), len(j), kind)) &&
               ok(hipEventRecord(ev[s], stream));
      };
      if (fetch(i, 0))
        for (int k = 0; i < pieces; i += workers, ++k) {
          const int s = k & 1;
          if (i + workers < pieces && !fetch(i + workers, s ^ 1)) break;
          if (!ok(hipEventSynchronize(ev[s]))) break;
          std::memcpy(h + at(i), b[s].p, len(i));
        }
    }
    const hipError_t f = b[0].wait(), g = b[1].wait();
    err[w] = e != hipSuccess ? e : f != hipSuccess ? f : g;
    for (auto x : ev)
      if (x) (void)hipEventDestroy(x);
  });
  for (int w = 0; w < workers; ++w)
    if (err[w] != hipSuccess) return err[w];
  return hipSuccess;
}

}  // namespace dgbgk
