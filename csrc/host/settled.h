// Memory that lives as long as the process, made where a call first needs it, and written before that call goes on. What the call's own stream
// would do is wrong twice: other streams would not wait for it, and on a stream that is capturing the fill would go into
// the graph, to run at its replays alone, and the memory would come from the graph's pool.
#pragma once
#include <ATen/ATen.h>
#include <c10/hip/HIPException.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <mutex>
#include <unordered_map>

namespace rt {

// While it lives the device's current stream is one that does not capture; settle() waits for what was given to it.
class Settled {
 public:
  explicit Settled(const at::Tensor& like)
      : relaxed_(hipStreamCaptureModeRelaxed), before_(c10::hip::getCurrentHIPStream(like.get_device())), side_(before_) {
    for (int tries = 0; side_ == before_ || capturing(side_); ++tries) {
      TORCH_CHECK(tries < 64, "no stream beside a capture");
      side_ = c10::hip::getStreamFromPool(false, like.get_device());
    }
    c10::hip::setCurrentHIPStream(side_);
  }
  ~Settled() { c10::hip::setCurrentHIPStream(before_); }
  Settled(const Settled&) = delete;
  Settled& operator=(const Settled&) = delete;
  void settle() { C10_HIP_CHECK(hipStreamSynchronize(side_.stream())); }

 private:
  static bool capturing(const c10::hip::HIPStream& s) {
    hipStreamCaptureStatus status;
    C10_HIP_CHECK(hipStreamIsCapturing(s.stream(), &status));
    return status != hipStreamCaptureStatusNone;
  }
  c10::hip::HIPStreamCaptureModeGuard relaxed_;
  c10::hip::HIPStream before_, side_;
};

// 4 KiB of zeros of a device: what products read in place of rows and columns that are not there
inline const at::Tensor& zero_page(const at::Tensor& like) {
  static std::mutex mu;
  static auto* map = new std::unordered_map<int, at::Tensor>();
  std::lock_guard<std::mutex> g(mu);
  auto it = map->find(like.get_device());
  if (it == map->end()) {
    Settled settled(like);
    at::Tensor page = at::zeros({2048}, like.options().dtype(at::kBFloat16));
    settled.settle();
    it = map->emplace(like.get_device(), page).first;
  }
  return it->second;
}

}  // namespace rt
