"""The memory contexts keep between calls (ast_memory.h) on the CPU, with
stand-ins for the HIP allocator: a device of 1000 MiB whose allocations fail
beyond that.  What one context keeps is given up for an allocation that would
fail, its own or another context's of the device; the bound, the reuse and the
trimming; takes and gives from several threads; under the address sanitizer."""
import subprocess

from asteroid_amd import build

PROGRAM = r"""
#include <cassert>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum { hipHostMallocDefault = 0 };
static std::mutex mu;
static thread_local int device = 0;
static size_t used[2] = {0, 0};
static std::map<void*, std::pair<int, size_t>> live;
static constexpr size_t MIB = (size_t)1 << 20, HAVE = 1000 * MIB;
static hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  if (used[device] + n > HAVE) return hipErrorOutOfMemory;
  *p = malloc(1);
  live[*p] = {device, n};
  used[device] += n;
  return hipSuccess;
}
static hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = live.find(p);
  assert(it != live.end());
  used[it->second.first] -= it->second.second;
  live.erase(it);
  free(p);
  return hipSuccess;
}
static hipError_t hipHostMalloc(void** p, size_t n, int) { *p = malloc(n); return hipSuccess; }
static hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
static hipError_t hipGetLastError() { return hipSuccess; }
#include "ast_memory.h"

// A block of n MiB taken and given back: it is kept.
static void keep(Memory& m, size_t n) {
  void* p;
  size_t cap;
  assert(m.take(n * MIB, &p, &cap) == hipSuccess && cap == n * MIB);
  m.give(p, cap);
}

// Closed after main, by the destructor of an object older than the registry.
struct Late {
  Memory* m = nullptr;
  ~Late() {
    if (m) m->close();
    delete m;
  }
} late;

int main() {
  Memory a, b, c;
  a.open(0);
  b.open(0);
  device = 1;
  c.open(1);
  keep(c, 100);
  device = 0;
  // bound and reuse
  keep(a, 200);
  assert(a.kept == 200 * MIB && used[0] == 200 * MIB);
  keep(a, 90);  // beyond the bound (and too small for the kept block): released
  assert(a.kept == 200 * MIB && used[0] == 200 * MIB);
  void *p, *q;
  size_t cap;
  assert(a.take(150 * MIB, &p, &cap) == hipSuccess && cap == 200 * MIB && a.kept == 0);
  a.give(p, cap);
  // an allocation of the context itself, then of another one, that needs what is kept
  assert(a.alloc(&p, 900 * MIB) == hipSuccess && a.kept == 0 && used[0] == 900 * MIB);
  hipFree(p);
  keep(a, 200);
  keep(b, 50);
  assert(used[0] == 250 * MIB);
  assert(b.alloc(&p, 900 * MIB) == hipSuccess && a.kept == 0 && b.kept == 0);
  assert(c.kept == 100 * MIB);  // the other device's
  assert(b.alloc(&q, 200 * MIB) == hipErrorOutOfMemory && q == nullptr);
  assert(b.take(200 * MIB, &q, &cap) == hipErrorOutOfMemory && q == nullptr);
  {
    Scratch s(b);
    s.reserve<double>((size_t)25 << 20);
    assert(s.take() == hipErrorOutOfMemory);
  }
  hipFree(p);
  // trim, oldest first
  keep(a, 60);
  assert(a.take(10 * MIB, &p, &cap) == hipSuccess && a.take(20 * MIB, &q, &cap) == hipSuccess);
  a.give(p, 10 * MIB);
  a.give(q, 20 * MIB);
  assert(a.kept == 90 * MIB);
  a.trim(40 * MIB);
  assert(a.kept == 30 * MIB && used[0] == 30 * MIB);
  a.trim(0);
  assert(a.kept == 0 && used[0] == 0);
  // threads: each context its own, allocations that fail now and then among them
  auto work = [](Memory* m, unsigned seed) {
    for (int i = 0; i < 4000; ++i) {
      seed = seed * 1664525u + 1013904223u;
      const size_t n = (size_t)(1 + (seed >> 8) % 120) * MIB;
      void* p;
      size_t cap;
      if (i % 7 == 0) {
        if (m->alloc(&p, 4 * n) == hipSuccess) hipFree(p);
      } else if (m->take(n, &p, &cap) == hipSuccess) {
        assert(cap >= n);
        m->give(p, cap);
      }
      assert(m->kept <= Memory::KEEP_BYTES);
    }
  };
  std::thread t1(work, &a, 1u), t2(work, &b, 2u);
  t1.join();
  t2.join();
  assert(a.pinned(Memory::PIN_BYTES + 1) == nullptr && a.pinned(1) && a.pinned(7) == a.pin);
  a.close();
  b.close();
  assert(used[0] == 0 && used[1] == 100 * MIB);
  c.close();
  assert(live.empty());
  late.m = new Memory;
  late.m->open(0);
  puts("memory ok");
}
"""


def test_kept_memory_is_bounded_and_given_up(tmp_path):
    src, exe = tmp_path / "memory.cpp", tmp_path / "memory"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-g", "-O1", "-pthread", "-fsanitize=address,undefined", "-I", build.CSRC,
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("memory ok"), r.stdout[-3000:]


def test_every_allocation_can_have_what_is_kept():
    with open(build.CSRC + "/ast_capi.hip") as f:
        assert "hipMalloc(" not in f.read()  # all go through Memory::alloc
