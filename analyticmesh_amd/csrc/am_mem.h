// Memory blocks kept between contexts.
//
// A context (one call of a training loop makes and drops one) needs some 60
// buffers, grown as its march grows: hipMalloc takes 0.1 to 0.4 ms whatever the
// size, hipFree as much and a wait for the device, pinned memory more: the
// 4x128 training step, which makes a context a step, took 51 ms and takes 32
// so.  Freed blocks therefore wait here for the next context: bounded (4 GiB of device memory, 256 MiB pinned),
// given back to the device when eight contexts have ended without using them,
// when the bound is passed (oldest first), when an allocation fails or the device is
// short of memory, or by am_trim_memory().  Contexts that end are what ages them: the
// blocks of a process's last ones stay until that call or the process's end.
// A block is given only when no work on it is pending (its stream has been
// waited for), so any stream may take it next.  Safe from several threads.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

namespace am {

enum MemKind { MEM_DEVICE = 0, MEM_PINNED, MEM_COHERENT, MEM_KINDS };

struct MemPool {
  struct Block {
    void* p;
    size_t bytes;
    int dev;
    long long epoch;
  };
  std::mutex m;
  std::vector<Block> kept[MEM_KINDS];   // oldest first
  size_t total[MEM_KINDS] = {0};
  long long epoch = 0;

  static MemPool& get() {
    static MemPool* pool = new MemPool();   // outlives every context (the runtime frees at process end)
    return *pool;
  }
  static size_t bound(int kind) { return kind == MEM_DEVICE ? (size_t)4 << 30 : (size_t)256 << 20; }
  // Sizes in eighths of a power of two, so that similar requests meet the same blocks.
  static size_t rounded(size_t bytes) {
    size_t step = 512;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
  }
  static hipError_t fresh(int kind, void** p, size_t bytes) {
    switch (kind) {
      case MEM_DEVICE: return hipMalloc(p, bytes);
      case MEM_PINNED: return hipHostMalloc(p, bytes, hipHostMallocDefault);
      default: return hipHostMalloc(p, bytes, hipHostMallocMapped | hipHostMallocCoherent);
    }
  }
  static void drop(int kind, const Block& b) {
    if (kind == MEM_DEVICE) (void)hipFree(b.p);
    else (void)hipHostFree(b.p);
  }
  // A block of at least `bytes` on the current device; *got its size.
  hipError_t take(int kind, size_t bytes, void** p, size_t* got) {
    bytes = rounded(std::max<size_t>(bytes, 1));
    int dev = 0;
    (void)hipGetDevice(&dev);
    {
      std::lock_guard<std::mutex> lock(m);
      std::vector<Block>& k = kept[kind];
      size_t best = k.size();
      for (size_t i = 0; i < k.size(); ++i)
        if (k[i].dev == dev && k[i].bytes >= bytes && k[i].bytes <= bytes + bytes / 4 &&
            (best == k.size() || k[i].bytes < k[best].bytes))
          best = i;
      if (best < k.size()) {
        *p = k[best].p;
        *got = k[best].bytes;
        total[kind] -= k[best].bytes;
        k.erase(k.begin() + best);
        return hipSuccess;
      }
    }
    hipError_t e = fresh(kind, p, bytes);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      trim(kind, 0, -1);
      e = fresh(kind, p, bytes);
    }
    *got = bytes;
    return e;
  }
  // Nothing that uses the block may be pending.
  void give(int kind, void* p, size_t bytes, int dev) {
    bool in = true;
    {
      std::lock_guard<std::mutex> lock(m);
      try {
        kept[kind].push_back(Block{p, bytes, dev, epoch});
        total[kind] += bytes;
      } catch (const std::bad_alloc&) {
        in = false;
      }
    }
    if (!in) drop(kind, Block{p, bytes, dev, 0});
    trim(kind, bound(kind), -1);
  }
  // Frees kept blocks, oldest first, down to `most` bytes, and those given before epoch `since`.
  void trim(int kind, size_t most, long long since) {
    for (;;) {
      Block b;
      {
        std::lock_guard<std::mutex> lock(m);
        std::vector<Block>& k = kept[kind];
        if (k.empty() || !(total[kind] > most || k[0].epoch < since)) return;
        b = k[0];
        total[kind] -= b.bytes;
        k.erase(k.begin());
      }
      drop(kind, b);
    }
  }
  // A context has ended.
  void age() {
    long long now;
    {
      std::lock_guard<std::mutex> lock(m);
      now = ++epoch;
    }
    for (int k = 0; k < MEM_KINDS; ++k) trim(k, bound(k), now - 8);
  }
  void clear() {
    for (int k = 0; k < MEM_KINDS; ++k) trim(k, 0, -1);
  }
};

// One block, given back when it goes.  Giving back waits for the device first, as
// hipFree does, unless the thread has done so for a whole context (MemQuiet); a
// block that cannot be waited for is freed instead of kept.
struct Mem {
  void* p = nullptr;
  size_t bytes = 0;
  int dev = 0, kind = MEM_DEVICE;
  Mem() = default;
  Mem(const Mem&) = delete;
  Mem& operator=(const Mem&) = delete;
  Mem(Mem&& o) noexcept { swap(o); }
  Mem& operator=(Mem&& o) noexcept {
    if (this != &o) {
      release();
      swap(o);
    }
    return *this;
  }
  ~Mem() { release(); }
  void swap(Mem& o) noexcept {
    std::swap(p, o.p);
    std::swap(bytes, o.bytes);
    std::swap(dev, o.dev);
    std::swap(kind, o.kind);
  }
  hipError_t take(int k, size_t n) {
    release();
    kind = k;
    (void)hipGetDevice(&dev);
    const hipError_t e = MemPool::get().take(k, n, &p, &bytes);
    if (e != hipSuccess) {
      p = nullptr;
      bytes = 0;
    }
    return e;
  }
  static int& quiet() {
    static thread_local int n = 0;
    return n;
  }
  void release() {
    if (!p) return;
    int cur = -1;
    const bool here = hipGetDevice(&cur) == hipSuccess && cur == dev;
    if (here && (quiet() || hipDeviceSynchronize() == hipSuccess)) MemPool::get().give(kind, p, bytes, dev);
    else MemPool::drop(kind, MemPool::Block{p, bytes, dev, 0});
    p = nullptr;
    bytes = 0;
  }
};

// Around a context's end: one wait for the device instead of one per block.
struct MemQuiet {
  bool on;
  MemQuiet() : on(hipDeviceSynchronize() == hipSuccess) { Mem::quiet() += on; }
  ~MemQuiet() { Mem::quiet() -= on; }
};

}  // namespace am
