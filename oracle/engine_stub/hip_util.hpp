#pragma once
// Test infrastructure: the few engine types that miso_amd/engine/attention.{hpp,hip} use (device
// buffers here; weights.hpp, gguf.hpp beside it), written to their interface so that the drop-in
// can be built and run where the engine is not at hand.

#include <hip/hip_runtime.h>

#include <cstddef>
#include <stdexcept>
#include <utility>
#include <vector>

#define MISO_HIP_CHECK(call)                                             \
  do {                                                                   \
    if (const hipError_t err_ = (call); err_ != hipSuccess)              \
      throw std::runtime_error(hipGetErrorString(err_));                 \
  } while (0)

namespace miso {

template <class T>
class DeviceBuffer {
 public:
  DeviceBuffer() = default;
  explicit DeviceBuffer(std::size_t n) : n_(n) {
    if (n != 0)
      MISO_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&p_), n * sizeof(T)));
  }
  explicit DeviceBuffer(const std::vector<T>& v) : DeviceBuffer(v.size()) {
    if (n_ != 0)
      MISO_HIP_CHECK(hipMemcpy(p_, v.data(), n_ * sizeof(T), hipMemcpyHostToDevice));
  }
  DeviceBuffer(DeviceBuffer&& o) noexcept : p_(std::exchange(o.p_, nullptr)), n_(o.n_) {}
  DeviceBuffer& operator=(DeviceBuffer&& o) noexcept {
    std::swap(p_, o.p_);
    std::swap(n_, o.n_);
    return *this;
  }
  ~DeviceBuffer() {
    if (p_ != nullptr)
      (void)hipFree(p_);
  }
  T* data() { return p_; }
  const T* data() const { return p_; }
  std::size_t size() const { return n_; }

 private:
  T* p_ = nullptr;
  std::size_t n_ = 0;
};

}  // namespace miso
