// The host framework's tensors from C++, without its headers (they are included by torch_bridge.cc alone) and without a Python
// call per property: a call of an operator with five tensors spent 6 us in the Python code that read them and 3 us in the
// one that allocated its result; 1 us and 1 us this way.
#ifndef MS_CUSTOM_OPS_FRAMEWORK_TORCH_BRIDGE_H_
#define MS_CUSTOM_OPS_FRAMEWORK_TORCH_BRIDGE_H_

#include <Python.h>

#include <cstddef>
#include <cstdint>

namespace ms_custom_ops {
struct TorchTensorView {
  void *data{nullptr};
  int type_id{0};            // MindSpore TypeId, 0 for a dtype without one
  bool on_gpu{false};
  size_t dims{0};
  const int64_t *sizes{nullptr};     // valid while the tensor lives and keeps its shape
  const int64_t *strides{nullptr};
};
// 1: *view is filled; 0: not a torch.Tensor; -1: a Python error is set.  The GIL is held.
int ViewTorchTensor(PyObject *object, TorchTensorView *view);
// torch.empty(sizes, dtype, device="cuda") on the current device: a new reference and its address, or nullptr with a Python error set
PyObject *NewTorchTensor(int type_id, const int64_t *sizes, size_t dims, void **data);
// index of the current GPU, or -1 with a Python error set
int CurrentTorchDevice();
}  // namespace ms_custom_ops
#endif  // MS_CUSTOM_OPS_FRAMEWORK_TORCH_BRIDGE_H_
