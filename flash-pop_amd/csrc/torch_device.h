// What the PyTorch ops ask about the device: whether a tensor is on it, its current stream, whether that stream is recording a
// HIP graph.  (Included by name through the include path: the CPU tests put a stand-in before it.)
#pragma once
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

namespace fpt {

inline bool on_device(const at::Tensor& t) { return t.is_cuda(); }
inline void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
inline bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

}  // namespace fpt
