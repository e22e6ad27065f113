// Deferred stage timing on one HIP stream: events are recorded between
// launches without waiting, and resolved once when the stream has drained,
// so timing adds no host round trip to a level.
#pragma once
#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>
#include <vector>

namespace am {

enum TimerSlot { T_CHAIN64 = 0, T_RAY64, T_SCAN64, T_GEMM, T_WALK, T_INSERT, T_VERT64, T_NEWTON, T_SLOTS };

// Stage times of a march taken on the device: the first thread of a stage's
// first kernel charges the time since the last mark to the stage that was
// running (kernels of a stream run one after another).  No events between the
// launches (each cost about 4 us of the stream's time), and the same inside a
// captured graph.  Ticks of wall_clock64(): 100 MHz.
struct StageClock {
  unsigned long long acc[T_SLOTS + 1];   // the last entry: between levels
  unsigned long long last;
  unsigned long long slot;
};
constexpr double kStageTickMs = 1e-5;
__device__ __forceinline__ void stage_mark_now(StageClock* c, int slot) {
  const unsigned long long t = wall_clock64();
  c->acc[c->slot] += t - c->last;
  c->last = t;
  c->slot = (unsigned long long)slot;
}
__device__ __forceinline__ void stage_mark(StageClock* c, int slot) {
  if (c && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) stage_mark_now(c, slot);
}

struct StageTimer {
  std::vector<hipEvent_t> pool;
  size_t used = 0;
  struct Span {
    size_t a, b;
    int slot;
  };
  std::vector<Span> spans;
  double acc[T_SLOTS] = {0};
  bool enabled = true;   // off: mark() and span() do nothing

  static void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e) + " in " + what);
  }
  // Record an event on `st`; returns its index for span().
  size_t mark(hipStream_t st) {
    if (!enabled) return 0;
    if (used == pool.size()) {
      hipEvent_t e;
      check(hipEventCreate(&e), "hipEventCreate");
      pool.push_back(e);
    }
    check(hipEventRecord(pool[used], st), "hipEventRecord");
    return used++;
  }
  void span(size_t a, size_t b, int slot) {
    if (enabled) spans.push_back({a, b, slot});
  }
  // The stream must have drained (or the events completed).
  void resolve() {
    for (const Span& s : spans) {
      float ms = 0;
      check(hipEventElapsedTime(&ms, pool[s.a], pool[s.b]), "hipEventElapsedTime");
      acc[s.slot] += ms;
    }
    spans.clear();
    used = 0;
  }
  void reset() {
    spans.clear();
    used = 0;
    for (double& a : acc) a = 0;
  }
  void release() {
    for (hipEvent_t e : pool) (void)hipEventDestroy(e);
    pool.clear();
    reset();
  }
};

}  // namespace am
