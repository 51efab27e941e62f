"""The pool of released device blocks (monolis_amd/csrc/mh_pool.hpp): on the CPU over an allocator with a
budget, on the GPU what monolis_hip_trim gives back."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include <thread>
#include <vector>
#include "mh_pool.hpp"
using namespace mh;
// A device of `left` bytes: blocks are 1-byte host allocations that remember their size.
struct Mem {
  size_t left = 0;
  std::map<void*, size_t> live;
  std::mutex mu;
};
static Mem M;
struct Fake {
  bool alloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lk(M.mu);
    if (bytes > M.left) return false;
    *p = std::malloc(1);
    M.live[*p] = bytes;
    M.left -= bytes;
    return true;
  }
  void free(void* p) {
    std::lock_guard<std::mutex> lk(M.mu);
    if (!M.live.count(p)) std::abort();
    M.left += M.live[p];
    M.live.erase(p);
    std::free(p);
  }
};
constexpr size_t KB = 1024, MB = KB * KB, GB = MB * KB;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
"""


def _run(tmp_path, body, flags=()):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(HEAD + "int main() {\n" + body + "\nreturn 0;\n}\n")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", *flags, "-I", os.path.join(ROOT, "monolis_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_blocks_are_reused_bounded_and_given_back(tmp_path):
    _run(tmp_path, r"""
  M.left = 100 * GB;
  BlockPool<Fake> P(4 * GB);
  void *a, *b;
  size_t ca, cb;
  CHECK(P.alloc(&a, 3 * MB + 7, 0, &ca) && ca >= 3 * MB + 7 && ca <= 4 * MB);
  P.free(a, ca);
  CHECK(P.alloc(&b, 3 * MB, 0, &cb) && b == a && cb == ca);     // a block a quarter larger serves
  P.free(b, cb);
  CHECK(P.alloc(&b, 1 * MB, 0, &cb) && b != a);                 // one three times as large does not
  P.free(b, cb);
  CHECK(P.alloc(&b, 3 * MB, 1, &cb) && b != a && cb == 0);      // another device: never kept
  P.free(b, cb);
  CHECK(M.live.size() == 2);
  std::vector<std::pair<void*, size_t>> v(7);
  for (auto& q : v) CHECK(P.alloc(&q.first, 1 * GB, 0, &q.second));
  for (auto& q : v) P.free(q.first, q.second);
  size_t held = 0;
  for (auto& q : M.live) held += q.second;
  CHECK(held <= 4 * GB);
  CHECK(P.trim() == held && M.live.empty() && M.left == 100 * GB && P.trim() == 0);
""")


def test_what_the_pool_holds_is_given_to_any_allocation_that_needs_it(tmp_path):
    _run(tmp_path, r"""
  M.left = 10 * GB;
  BlockPool<Fake> P(4 * GB);
  void *a, *b, *u;
  size_t ca, cb;
  CHECK(P.alloc(&a, 3 * GB, 0, &ca));
  P.free(a, ca);
  CHECK(M.left == 7 * GB);
  CHECK(P.alloc_outside(&u, 8 * GB) && M.left == 2 * GB);       // a user's buffer
  CHECK(!P.alloc_outside(&b, 8 * GB));
  Fake().free(u);
  CHECK(P.alloc(&a, 3 * GB, 0, &ca));
  P.free(a, ca);
  CHECK(P.alloc(&b, 8 * GB, 0, &cb));                           // the library's own
  P.free(b, cb);
  CHECK(M.left == 10 * GB && M.live.empty());                   // larger than the limit: not kept
""")


def test_rounding_refuses_nothing_that_fits(tmp_path):
    _run(tmp_path, r"""
  M.left = 200 * GB;
  BlockPool<Fake> P(4 * GB);
  void *a, *b, *c;
  size_t ca, cb, cc;
  CHECK(P.alloc(&a, 196 * GB, 0, &ca) && M.left == 4 * GB);     // larger than any block kept: exactly its size
  CHECK(P.alloc(&b, 3 * GB - 1, 0, &cb) && M.left == 1 * GB);   // rounded up
  CHECK(P.alloc(&c, 1 * GB - 3, 0, &cc));
  P.free(c, cc);
  P.trim();
  M.left -= 5;
  CHECK(M.left == 1 * GB - 5);
  CHECK(P.alloc(&c, 1 * GB - 6, 0, &cc));                       // its rounded size no longer fits
  P.free(c, cc);
  P.free(b, cb);
  P.free(a, ca);
  P.trim();
  CHECK(M.live.empty() && M.left == 200 * GB - 5);
""")


def test_threads_share_the_pool(tmp_path):
    _run(tmp_path, r"""
  M.left = 1000 * GB;
  BlockPool<Fake> P(64 * MB);
  std::mutex mu;
  std::set<void*> used;
  bool bad = false;
  auto work = [&](unsigned seed) {
    for (int i = 0; i < 2000; ++i) {
      seed = seed * 1664525u + 1013904223u;
      void* p;
      size_t cap;
      if (!P.alloc(&p, (seed >> 8) % (4 * MB) + 1, 0, &cap)) bad = true;
      { std::lock_guard<std::mutex> lk(mu); if (!used.insert(p).second) bad = true; }
      { std::lock_guard<std::mutex> lk(mu); used.erase(p); }
      P.free(p, cap);
      if (i % 500 == 0) P.trim();
    }
  };
  std::vector<std::thread> t;
  for (unsigned k = 0; k < 6; ++k) t.emplace_back(work, k + 1);
  for (auto& x : t) x.join();
  CHECK(!bad);
  P.trim();
  CHECK(M.live.empty());
""")


@pytest.mark.gpu
def test_trim_gives_the_memory_back(hip):
    from monolis_amd import api, workloads as W

    def left():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0   # of the runtime it is linked with
        return free.value

    api.trim()
    free0 = left()
    dm = api.DeviceMatrix(W.stencil27_bcsr3(24, seed=1))
    del dm
    kept = free0 - left()
    assert kept >= 24 ** 3 * 200 * 8
    assert api.trim() >= 24 ** 3 * 200 * 8
    assert free0 - left() < kept // 2
    dm = api.DeviceMatrix(W.poisson7(12))                      # and it goes on from there
    b, x = api.DeviceBuffer.from_numpy(W.uniform_vector(dm.mat.n, seed=1)), api.DeviceBuffer(dm.mat.n)
    prm = api.Prm().quiet()
    dm.solve(b, x, prm)
    assert prm.Iarray[api.MONOLIS_PRM_I_IERR] == 0
