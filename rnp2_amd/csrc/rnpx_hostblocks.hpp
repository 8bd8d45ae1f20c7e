// rnpx_hostblocks.hpp -- the server's copies of its requests and the host memory
// that they are in.  Plain C++ over a pair of pin/unpin functions: a CPU test
// compiles this file.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace rnpx {

// dst (m x n, leading dimension m) = src (leading dimension lds): large
// matrices split over host threads by columns (one thread copies a few GB/s;
// a 8192 x 4096 request is 268 MB; a thread's start is worth about 4 MB).  A
// thread that the system refuses leaves its columns to this one: the caller is
// a C entry, where nothing may be thrown.
template <class Thread>
void copy_columns(double* dst, const double* src, size_t m, size_t n, size_t lds) {
  const size_t bytes = sizeof(double) * m * n;
  const size_t hw = std::max(1u, std::thread::hardware_concurrency());
  const size_t nt = std::min<size_t>({(size_t)8, hw, n, std::max<size_t>(1, bytes >> 22)});
  const size_t per = (n + nt - 1) / nt;
  auto part = [&](size_t q) {
    for (size_t j = std::min(n, q * per); j < std::min(n, (q + 1) * per); ++j)
      std::memcpy(dst + j * m, src + j * lds, sizeof(double) * m);
  };
  Thread th[8];
  for (size_t q = 1; q < nt; ++q) {
    try {
      th[q] = Thread(part, q);
    } catch (const std::system_error&) {
      part(q);
    }
  }
  part(0);
  for (Thread& x : th)
    if (x.joinable()) x.join();
}

struct HostBlock {
  double* p = nullptr;
  size_t bytes = 0;
  bool pinned = false;
};

// Pinned blocks that go back to a list when a request is done, so that a submit
// neither faults fresh pages in nor clears them before the copy, and the
// transfer to the device is one asynchronous DMA.  At most `cap` bytes in all, in
// use or idle; idle ones are given back by trim() and at the end.  A request beyond
// that (or where pinned memory is refused) takes ordinary memory.
// Pin: bool pin(void** p, size_t bytes), void unpin(void* p).
template <class Pin>
class HostBlocks {
 public:
  explicit HostBlocks(size_t cap) : cap_(cap) {}
  HostBlocks(const HostBlocks&) = delete;
  HostBlocks& operator=(const HostBlocks&) = delete;
  ~HostBlocks() { trim(); }

  // pin: false for memory that no transfer reads.
  HostBlock take(size_t bytes, bool pin) {
    // sizes in eighths of a power of two, 64 KB at least: a block serves
    // requests down to half its size
    size_t unit = (size_t)64 << 10;
    while (unit * 16 < bytes) unit *= 2;
    const size_t want = std::max<size_t>((size_t)64 << 10, (bytes + unit - 1) / unit * unit);
    std::vector<HostBlock> drop;
    bool room = false;
    if (pin) {
      std::lock_guard<std::mutex> lk(mu_);
      size_t best = idle_.size(), idle = 0;
      for (size_t i = 0; i < idle_.size(); ++i) {
        idle += idle_[i].bytes;
        if (idle_[i].bytes >= want && idle_[i].bytes <= 2 * want &&
            (best == idle_.size() || idle_[i].bytes < idle_[best].bytes))
          best = i;
      }
      if (best < idle_.size()) {
        HostBlock b = idle_[best];
        idle_.erase(idle_.begin() + (long)best);
        return b;
      }
      // room for a new one, if need be in place of idle blocks of other sizes, the
      // longest unused first -- and only if that makes room
      room = held_ - idle + want <= cap_;
      size_t n = 0;
      for (; room && held_ + want > cap_; ++n) {
        held_ -= idle_[n].bytes;
        drop.push_back(idle_[n]);
      }
      idle_.erase(idle_.begin(), idle_.begin() + (long)n);
      if (room) held_ += want;
    }
    // (the driver's calls, tens of milliseconds for a large block, outside the lock)
    for (HostBlock& b : drop) Pin::unpin(b.p);
    if (room) {
      void* p = nullptr;
      if (Pin::pin(&p, want)) return HostBlock{static_cast<double*>(p), want, true};
      std::lock_guard<std::mutex> lk(mu_);
      held_ -= want;
    }
    return HostBlock{static_cast<double*>(std::malloc(std::max<size_t>(bytes, 8))), bytes, false};
  }

  void give(HostBlock& b) {
    if (!b.p) return;
    if (b.pinned) {
      std::lock_guard<std::mutex> lk(mu_);
      idle_.push_back(b);
    } else {
      std::free(b.p);
    }
    b = HostBlock{};
  }

  // The idle blocks back to the system.
  void trim() {
    std::vector<HostBlock> drop;
    {
      std::lock_guard<std::mutex> lk(mu_);
      drop.swap(idle_);
      for (HostBlock& b : drop) held_ -= b.bytes;
    }
    for (HostBlock& b : drop) Pin::unpin(b.p);
  }

  size_t held() {
    std::lock_guard<std::mutex> lk(mu_);
    return held_;
  }

 private:
  const size_t cap_;
  std::mutex mu_;
  std::vector<HostBlock> idle_;  // in the order they were given back
  size_t held_ = 0;
};

}  // namespace rnpx
