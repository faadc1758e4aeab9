#pragma once
// Test infrastructure (see ../hip_util.hpp): the engine's quantised matrix and GEMM input.

#include <cstddef>
#include <cstdint>
#include <stdexcept>
#include <string>

#include "gguf.hpp"
#include "hip_util.hpp"

namespace miso {

struct QMatrix {
  gguf::GgmlType type;
  unsigned n, k;
  DeviceBuffer<std::uint8_t> data;
};

struct GemmInput {
  GemmInput(std::size_t max_tok, std::size_t max_k)
      : xh(max_tok * max_k), xs(max_tok * max_k / 32) {}
  DeviceBuffer<_Float16> xh;
  DeviceBuffer<float> xs;
  unsigned k = 0, n_tok = 0;
};

struct LoadStage;
inline QMatrix upload_qmatrix(const gguf::File&, const std::string& name, LoadStage*) {
  throw std::runtime_error("no " + name);
}
inline DeviceBuffer<float> upload_f32(const gguf::File&, const std::string& name, LoadStage*) {
  throw std::runtime_error("no " + name);
}

}  // namespace miso
