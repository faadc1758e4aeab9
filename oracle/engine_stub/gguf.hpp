#pragma once
// Test infrastructure (see hip_util.hpp): a file that holds nothing.

#include <stdexcept>
#include <string>

namespace miso::gguf {

enum class GgmlType { Q4_K, Q6_K };

struct File {
  template <class T>
  T get(const std::string& key) const {
    throw std::runtime_error("no " + key);
  }
};

}  // namespace miso::gguf
