// Forwards that gave up a bounded wait of theirs (encoder_few.hip). The kernel writes a word of pinned host memory, one a device, and the host
// looks at it without waiting for anything: at the next forward, and wherever the package has just waited for results.
#pragma once
#include <c10/hip/HIPException.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <hip/hip_runtime_api.h>

#include <cstring>
#include <mutex>

namespace rt {

constexpr int LOST_DEVICES = 64, LOST_STRIDE = 32;  // a word a line

// made by the first forward and kept: graphs write it by its address
inline unsigned* lost_word(int device) {
  static std::mutex mu;
  static unsigned* words = nullptr;
  TORCH_CHECK(device >= 0 && device < LOST_DEVICES, "device ", device);
  std::lock_guard<std::mutex> g(mu);
  if (!words) {
    c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
    void* p = nullptr;
    const size_t bytes = sizeof(unsigned) * LOST_DEVICES * LOST_STRIDE;
    C10_HIP_CHECK(hipHostMalloc(&p, bytes, hipHostMallocPortable | hipHostMallocMapped));
    std::memset(p, 0, bytes);
    words = (unsigned*)p;
  }
  return words + device * LOST_STRIDE;
}

inline void raise_lost(int device) {
  TORCH_CHECK(!__atomic_exchange_n(lost_word(device), 0u, __ATOMIC_RELAXED), "an encoder's forward on GPU ", device,
              " gave up waiting for rows of its own: embeddings that it returned are NaN");
}

}  // namespace rt
