// ibg_pinned.h — two pinned host buffers with the event that ends the use of
// each (ibg_closure_infer).
#pragma once
#include <hip/hip_runtime.h>

#include <stddef.h>

namespace ibg {

struct PinnedPair {
  float *buf[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};
  // Whatever of the two is not there yet: a call after one that failed half
  // way makes the rest.
  bool make(size_t bytes) {
    for (int b = 0; b < 2; ++b) {
      if (!buf[b] && hipHostMalloc((void **)&buf[b], bytes, hipHostMallocDefault) != hipSuccess) {
        buf[b] = nullptr;
        return false;
      }
      if (!done[b] && hipEventCreateWithFlags(&done[b], hipEventDisableTiming) != hipSuccess) {
        done[b] = nullptr;
        return false;
      }
    }
    return true;
  }
  void release() {
    for (int b = 0; b < 2; ++b) {
      if (buf[b]) (void)hipHostFree(buf[b]);
      if (done[b]) (void)hipEventDestroy(done[b]);
      buf[b] = nullptr;
      done[b] = nullptr;
    }
  }
};

}  // namespace ibg
