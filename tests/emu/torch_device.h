// CPU stand-in for the device queries of the PyTorch ops: tensors on the CPU, no stream, the capture flag of launch_emu.cpp.
#pragma once
#include <ATen/core/Tensor.h>

int fpk_stream_is_capturing(void* stream);

namespace fpt {

inline bool on_device(const at::Tensor& t) { return t.is_cpu(); }
inline void* stream() { return nullptr; }
inline bool capturing() { return fpk_stream_is_capturing(nullptr) != 0; }

}  // namespace fpt
