// Host-side operand checks: a kernel that is handed a host pointer faults the
// GPU, so wrappers refuse one first.
#pragma once

#include <torch/extension.h>

inline void on_gpu(std::initializer_list<c10::optional<torch::Tensor>> tensors) {
  for (const auto& t : tensors)
    TORCH_CHECK(!t.has_value() || t->is_cuda(), "all operands must be on the GPU");
}

// A contiguous tensor on 16 bytes, as wide and direct loads want it: itself, or a copy.
inline torch::Tensor on16(const torch::Tensor& t) {
  return (uintptr_t)t.data_ptr() % 16 ? t.clone() : t;
}
