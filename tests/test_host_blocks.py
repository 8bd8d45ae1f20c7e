"""The server's pinned request memory, with counting pin functions in a CPU
build: the cap holds, idle blocks are dropped only where that makes room (the
longest unused first), memory that no transfer reads is not pinned, trim() gives
every idle block back, and several threads share the list.  The copies into it are
whole where the system refuses threads."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rnp2_amd", "csrc")
MAIN = r"""
#include "rnpx_hostblocks.hpp"
#include <atomic>
#include <cstdio>
#include <thread>
static std::atomic<int> pins{0}, unpins{0};
static std::atomic<bool> refuse{false};
struct Fake {
  static bool pin(void** p, size_t n) { if (refuse) return false; ++pins; *p = std::malloc(n); return true; }
  static void unpin(void* p) { ++unpins; std::free(p); }
};
// a thread that cannot be had every other time
struct Scarce : std::thread {
  static int tries;
  Scarce() = default;
  Scarce(Scarce&&) = default;
  Scarce& operator=(Scarce&&) = default;
  template <class F> Scarce(F f, size_t q) : std::thread(start(), f, q) {}
  struct Run { template <class F> void operator()(F f, size_t q) { f(q); } };
  static Run start() {
    if (++tries % 2) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
    return Run();
  }
};
int Scarce::tries = 0;
template <class T> static bool copies(size_t m, size_t n, size_t lds) {
  std::vector<double> a(lds * n), b(m * n, -1.0);
  for (size_t i = 0; i < a.size(); ++i) a[i] = (double)i;
  rnpx::copy_columns<T>(b.data(), a.data(), m, n, lds);
  for (size_t j = 0; j < n; ++j)
    for (size_t i = 0; i < m; ++i)
      if (b[i + j * m] != a[i + j * lds]) return false;
  return true;
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s (pins %d unpins %d)\n", __LINE__, #x, pins.load(), unpins.load()); return 1; } } while (0)
int main() {
  using namespace rnpx;
  const size_t MB = 1 << 20;
  for (size_t n : {1, 2, 7, 9, 1000, 5000}) {
    CHECK(copies<std::thread>(1000, n, 1003));
    CHECK(copies<Scarce>(1000, n, 1003));
  }
  CHECK(Scarce::tries > 3);
  {
    HostBlocks<Fake> h(100 * MB);
    HostBlock a = h.take(30 * MB, true), b = h.take(30 * MB, true), c = h.take(30 * MB, true);
    CHECK(pins == 3 && a.pinned && b.pinned && c.pinned);
    h.give(a); h.give(b);
    // too large whatever is dropped: ordinary memory, nothing dropped
    HostBlock d = h.take(90 * MB, true);
    CHECK(!d.pinned && d.p && unpins == 0);
    h.give(d);
    HostBlock e = h.take(200 * MB, true);
    CHECK(!e.pinned && e.p && unpins == 0);
    h.give(e);
    // a smaller one reuses; half the size and less does not
    HostBlock f = h.take(20 * MB, true);
    CHECK(f.pinned && pins == 3 && unpins == 0 && f.bytes >= 30 * MB);
    // 8 MB fits beside them (no drop); 35 MB in place of the idle one
    HostBlock g = h.take(8 * MB, true);
    CHECK(g.pinned && pins == 4 && unpins == 0);
    HostBlock i = h.take(32 * MB, true);
    CHECK(i.pinned && pins == 5 && unpins == 1 && h.held() <= 100 * MB);
    // not pinned: no pin call
    HostBlock j = h.take(MB, false);
    CHECK(!j.pinned && j.p && pins == 5);
    h.give(c); h.give(f); h.give(g); h.give(i); h.give(j);
    h.trim();
    CHECK(unpins == 5 && h.held() == 0);
    refuse = true;
    HostBlock k = h.take(MB, true);
    CHECK(!k.pinned && k.p && h.held() == 0);
    h.give(k);
    refuse = false;
    std::thread t[4];
    for (int q = 0; q < 4; ++q)
      t[q] = std::thread([&h, q] {
        for (int r = 0; r < 2000; ++r) {
          HostBlock x = h.take(((size_t)1 << 16) * (1 + (r * 7 + q) % 90), true);
          x.p[0] = q;
          if (r % 97 == 0) h.trim();
          h.give(x);
        }
      });
    for (auto& x : t) x.join();
    CHECK(h.held() <= 100 * MB);
  }
  CHECK(pins == unpins);
  std::puts("ok");
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")
def test_blocks(tmp_path):
    src, exe = tmp_path / "blocks.cpp", tmp_path / "blocks"
    src.write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout

