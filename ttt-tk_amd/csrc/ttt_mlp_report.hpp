// Ints in host memory that the device writes when a wait gives up, so that after its own wait for the stream the host knows without
// a copy from the device (a second wait: forward of 2 pairs x 4 mini-batches 75.3 us with it, 62.8 us so).
#pragma once
#include <hip/hip_runtime_api.h>

#include <mutex>
#include <vector>

// One block, allocated at the first launch that needs one and kept for the process; word 0 collects the launches that nobody waits for,
// the others serve one waiting call each.  Where there is no such memory a waiting call copies its launch's status word, and
// a launch that nobody waits for takes one workgroup per (batch, head), which waits for nobody; the next call asks again.
struct ReportWords {
  static constexpr int WORDS = 64, STRIDE = 16;   // ints; a cache line each
  std::mutex mutex;
  int* block = nullptr;
  std::vector<int> unused;
  bool ready() {   // (mutex held)
    if (block == nullptr) {
      hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;   // the caller may be recording a graph
      (void)hipThreadExchangeStreamCaptureMode(&mode);
      void* p = nullptr;
      if (hipHostMalloc(&p, WORDS * STRIDE * sizeof(int), hipHostMallocPortable | hipHostMallocMapped) == hipSuccess) {
        block = static_cast<int*>(p);
        for (int i = 0; i < WORDS * STRIDE; i++) block[i] = 0;
        for (int i = 1; i < WORDS; i++) unused.push_back(i);
      } else {
        (void)hipGetLastError();
      }
      (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
    return block != nullptr;
  }
  int* collecting() {   // nullptr: none
    const std::lock_guard<std::mutex> lock(mutex);
    return ready() ? block : nullptr;
  }
  // Whether a launch whose workgroups wait for each other can say that one gave up.
  bool serves(bool host_waits) { return host_waits || collecting() != nullptr; }
  int* take() {   // nullptr: none, or none left
    const std::lock_guard<std::mutex> lock(mutex);
    if (!ready() || unused.empty()) return nullptr;
    int* const w = block + unused.back() * STRIDE;
    unused.pop_back();
    __atomic_store_n(w, 0, __ATOMIC_RELAXED);
    return w;
  }
  void give(int* w) {
    const std::lock_guard<std::mutex> lock(mutex);
    unused.push_back(static_cast<int>(w - block) / STRIDE);
  }
};
