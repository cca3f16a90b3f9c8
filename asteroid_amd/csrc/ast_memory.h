// ast_memory.h -- a context's device and pinned host memory between calls.
//
// An allocation and a release cost a call about 15 us each (a release waits
// for the device as well), three to fourteen of them a chi^2 batch or a job.
//  * blocks: device blocks given back by finished calls and jobs, taken again
//    by later ones of up to their size; at most KEEP_BYTES, the rest is
//    released.  A call gives its blocks back when nothing on the device uses
//    them any more.
//  * pin: pinned host memory that kernels read and write in place, for inputs
//    and results so small that a copy's latency is most of its time.
// What is kept is nobody's need: where an allocation on the device fails, of
// whichever context, the blocks that all contexts keep there are released
// and it is tried again.
//
// Calls on a context come from one thread at a time (the scheduler's while it
// serves); the lock is for other contexts' threads.
//
// Includes no HIP header: the includer has one (or, in a CPU test, its
// stand-ins for the few calls used here).
#pragma once
#include <algorithm>
#include <cstddef>
#include <mutex>
#include <utility>
#include <vector>

struct Memory {
  static constexpr size_t KEEP_BYTES = (size_t)256 << 20, PIN_BYTES = (size_t)4 << 20;
  std::vector<std::pair<size_t, void*>> blocks;
  size_t kept = 0;
  char* pin = nullptr;

  void open(int dev) {
    const std::lock_guard<std::mutex> lk(all_mu());
    device = dev;
    all().push_back(this);
  }
  void close() {
    {
      const std::lock_guard<std::mutex> lk(all_mu());
      release(0);
      all().erase(std::remove(all().begin(), all().end(), this), all().end());
    }
    if (pin) (void)hipHostFree(pin);
    pin = nullptr;
  }

  // hipMalloc on the context's device (the current one), with what is kept
  // there given up for it if it must be.
  hipError_t alloc(void** p, size_t bytes) {
    *p = nullptr;
    if (hipMalloc(p, bytes) == hipSuccess) return hipSuccess;
    (void)hipGetLastError();
    const std::lock_guard<std::mutex> lk(all_mu());
    for (Memory* m : all())
      if (m->device == device) m->release(0);
    *p = nullptr;
    return hipMalloc(p, bytes);
  }

  // A block of at least `bytes`: the smallest kept one that holds it, of at
  // most twice its size, else a new one.
  hipError_t take(size_t bytes, void** p, size_t* cap) {
    bytes = (bytes + 4095) & ~(size_t)4095;
    {
      const std::lock_guard<std::mutex> lk(all_mu());
      int best = -1;
      for (int k = 0; k < (int)blocks.size(); ++k)
        if (blocks[k].first >= bytes && blocks[k].first <= 2 * bytes &&
            (best < 0 || blocks[k].first < blocks[best].first))
          best = k;
      if (best >= 0) {
        *cap = blocks[best].first;
        *p = blocks[best].second;
        kept -= *cap;
        blocks.erase(blocks.begin() + best);
        return hipSuccess;
      }
    }
    *cap = bytes;
    return alloc(p, bytes);
  }
  void give(void* p, size_t cap) {
    if (!p) return;
    {
      const std::lock_guard<std::mutex> lk(all_mu());
      if (kept + cap <= KEEP_BYTES && blocks.size() < 64) {
        blocks.push_back({cap, p});
        kept += cap;
        return;
      }
    }
    (void)hipFree(p);
  }
  // Keep at most `most` bytes.
  void trim(size_t most) {
    const std::lock_guard<std::mutex> lk(all_mu());
    release(most);
  }

  // Pinned memory for `bytes`, or null (too many, or none to be had): the
  // caller copies instead.
  char* pinned(size_t bytes) {
    if (bytes > PIN_BYTES) return nullptr;
    if (!pin && hipHostMalloc((void**)&pin, PIN_BYTES, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      pin = nullptr;
    }
    return pin;
  }

 private:
  int device = -1;
  // Never destroyed: a program may close its contexts as it exits.
  static std::mutex& all_mu() {
    static std::mutex& m = *new std::mutex;
    return m;
  }
  static std::vector<Memory*>& all() {  // the open ones
    static std::vector<Memory*>& v = *new std::vector<Memory*>;
    return v;
  }
  // (with the lock) the oldest blocks first
  void release(size_t most) {
    size_t k = 0;
    for (; k < blocks.size() && kept > most; ++k) {
      (void)hipFree(blocks[k].second);
      kept -= blocks[k].first;
    }
    blocks.erase(blocks.begin(), blocks.begin() + k);
  }
};

// One device block of a call, given back at its end; carve() hands out its
// parts, in the order and sizes of the reserve() calls before it.
struct Scratch {
  Memory& mem;
  void* base = nullptr;
  size_t cap = 0, need = 0, at = 0;
  explicit Scratch(Memory& m) : mem(m) {}
  ~Scratch() { mem.give(base, cap); }
  static size_t padded(size_t bytes) { return (bytes + 255) & ~(size_t)255; }
  template <class T> void reserve(size_t n) { need += padded(n * sizeof(T)); }
  hipError_t take() { return mem.take(need ? need : 256, &base, &cap); }
  template <class T> T* carve(size_t n) {
    T* p = (T*)((char*)base + at);
    at += padded(n * sizeof(T));
    return p;
  }
};
